// C ABI of the ETD engine: plans (geometry, symbols, coefficient tables), transforms, stepping,
// graph capture.  Kernels live in k_*.hip; this file holds host logic only.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "engine.hpp"
#include "gfft.hpp"
#include "tfsm.h"

using namespace tfsm;

namespace tfsm {
thread_local hipEvent_t g_launch_ev[2] = {nullptr, nullptr};
}

// Workspace of tfsm_step_noalloc: a device array of fixed size, one copy per GPU, loaded with the
// code object and held until the process ends.  Host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (scratch_on_device below); the name itself is
// a host-side stand-in and never a device address.
static __device__ __align__(256) unsigned char scratch[TFSM_NOALLOC_SCRATCH_BYTES];

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
    return fail(TFSM_E_OOM, std::string(what) + ": out of device memory (" + hipGetErrorString(e) + ")");
  return fail(TFSM_E_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

// status of a HIP call as a TFSM code (0 on success), for code paths with a single exit
int launch_status(hipError_t e, const char* what) { return e == hipSuccess ? TFSM_OK : hip_fail(e, what); }

#define HIP_TRY(expr, what)               \
  do {                                    \
    hipError_t _e = (expr);               \
    if (_e != hipSuccess) return hip_fail(_e, what); \
  } while (0)

bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }
size_t roundup(size_t x, size_t m) { return (x + m - 1) / m * m; }

// fftfreq order of integer wavenumbers
int signed_k(int i, int n) { return i < (n + 1) / 2 ? i : i - n; }

// axis wavenumbers exactly as the reference forms them in float32:
// f = fl32(k) * fl32(1 / (n d)), d = length / n  (torch.fft.fftfreq, mesh.py:185-191)
// a = fl32(fl32(2 pi) * f)                        ((2j*pi*bf)^1, mesh.py:399-404)
void axis_table(int n, double length, std::vector<float>& a, std::vector<float>* f_out = nullptr) {
  const double d = length / n;
  const float s = (float)(1.0 / (n * d));
  const float two_pi = (float)(2.0 * M_PI);
  a.resize(n);
  if (f_out) f_out->resize(n);
  for (int i = 0; i < n; ++i) {
    const float f = (float)signed_k(i, n) * s;
    a[i] = two_pi * f;
    if (f_out) (*f_out)[i] = f;
  }
}

// low_pass_filter (mesh.py:443-461): keep |f| <= max|f| * rate, in float32; returns max kept |k|
int dealias_kmax(int n, double length, double rate) {
  std::vector<float> a, f;
  axis_table(n, length, a, &f);
  float fmax = 0.f;
  for (float v : f) fmax = std::fabs(v) > fmax ? std::fabs(v) : fmax;
  const float thr = fmax * (float)rate;
  int kmax = -1;
  for (int i = 0; i < n; ++i) {
    const int k = std::abs(signed_k(i, n));
    const bool masked = std::fabs(f[i]) > thr;
    if (!masked && k > kmax) kmax = k;
  }
  // the kept set must be {|k| <= kmax} for the engine's index-range mask
  for (int i = 0; i < n; ++i) {
    const int k = std::abs(signed_k(i, n));
    const bool masked = std::fabs(f[i]) > thr;
    if ((k <= kmax) == masked) return -2;
  }
  return kmax;
}

}  // namespace

struct tfsm_plan {
  int device = 0;  // HIP device current at tfsm_plan_create (its tables live there)
  int D = 0, n[3] = {1, 1, 1}, B = 0, C = 0;
  double len[3] = {0, 0, 0};
  int H = 0, P = 0;
  size_t modes = 0;  // complex elements of one [N...] block in half-spectrum layout
  int term = TERM_NONE;
  bool ks_mean = false;  // KSConvection(remove_mean=True): the batch mean of the product is removed
  float coef_t = 0.f;
  double rate = 2.0 / 3.0;
  int kmax[3] = {0, 0, 0};
  int nlin = 0;
  int lin_kind[4] = {0, 0, 0, 0};
  int lin_dim[4] = {0, 0, 0, 0}, lin_order[4] = {0, 0, 0, 0};
  bool cplx = false;        // complex L (odd-order SpatialDerivative): complex symbol and tables
  float2* Lc = nullptr;     // [Bc][modes]
  float2* coefc = nullptr;  // [Bc][NCOEF][modes]
  bool per_len = false;  // 1D plan with per-sample lengths (axis tables per row)
  int Bc = 1;
  float2* tw[3][4] = {};  // [axis][radix-plan variant]
  float* kv[3] = {nullptr, nullptr, nullptr};
  size_t kv_bstride = 0;
  float* L = nullptr;
  float* coef = nullptr;
  float4* cpk = nullptr;  // packed per-mode coefficients of the current scheme
  float* c5t = nullptr;   // SETDRK4's c5 per mode (read alone by the third evaluation)
  float2* ck01 = nullptr; // SETDRK4's [E2, c1] per mode (first and second evaluations)
  float* c6t = nullptr;   // SETDRK4's c6 per mode (last evaluation)
  int scheme = -1;
  double dt = 0.0;
  int n_points = 16;
  double radius = 1.0;
  float2* src = nullptr;
  int srcB = 0, srcC = 0;
  unsigned char* src_cols = nullptr;  // 2D: [P] 1 where a source mode of last-axis column k is nonzero
  uint32_t src_bits[Col2Args::SRC_BIT_WORDS] = {};  // the same flags as bits (P <= 544)
  bool src_bits_ok = false;
  int V = 16;        // column tile of the fused 2D column kernel
  int col_var = 0;   // radix-plan variant of the column transforms
  int row_var = 0;   // radix-plan variant of the row transforms
  int row_wg = 256;  // row-kernel workgroup size
  int sub_batch = 0; // samples stepped together through all steps (0 = whole batch)
  int nstreams = 1;  // > 1: sub-batch k runs on stream k % nstreams (0: the caller's, i: aux[i - 1])
  bool persistent = false;  // 2D: step with the persistent per-sample kernel k2_run
  hipStream_t aux[TFSM_MAX_STREAMS - 1] = {};
  hipEvent_t ev_fork = nullptr, ev_join[TFSM_MAX_STREAMS - 1] = {};
  int PF = 0, NF = 0;
  int K1 = 0;  // 3D: kept ky values (2 kmax1 + 1)
  size_t off_A1 = 0, off_A2 = 0, off_P = 0, off_G = 0, off_G2 = 0, ws_bytes = 0;
  size_t off_DC = 0;              // KSConvection: batch mean of the product DC (one complex value)
  size_t off_S = 0, off_N = 0;    // 1D KSConvection: stage spectrum and raw product spectrum
  // long 1D meshes (k_long1d.hip): N = l1 l2, field and product pitch PF
  int l1 = 0, l2 = 0;
  float2 *ltw1 = nullptr, *ltw2 = nullptr, *ltw4 = nullptr;
  std::vector<void*> allocs;
  // adjoint (tfsm_adjoint_prepare)
  float* dcoef = nullptr;  // [Bc][3][modes]
  float* sym = nullptr;    // [modes]
  int adj_term = -2;       // linear term whose coefficient gets a gradient (-1 none; -2 not prepared)
  int adj_scheme = -1;
  // unfused path (k_general.hip): stepping without the fused kernels
  bool general = false;    // no fixed-size fused kernels step the plan (genf: those of run-time lengths; else unfused)
  bool fused_ok = false;   // the fused kernels cover this plan (the unfused path is then optional)
  GAxis gax[3];            // general-length FFT tables of the axes without fixed-size kernels
  float2* gtmp = nullptr;  // four-step scratch of those axes
  float2* force = nullptr;  // NSPressureConvection's external force spectrum [forceB][forceC][modes]
  int forceB = 0, forceC = 0;
  // general plans that step on the fused kernels of run-time lengths (k_genfused.hip): 2D (gf_row, gf_col: that
  // axis takes the run-time kernel, the other one its fixed-size kernel) or the persistent 1D stepper
  // (genf: taken now; genf_ok: the plan has them, set_general(1) leaves them aside)
  bool genf = false, genf_ok = false, gf_row = false, gf_col = false;
  size_t ws_fused = 0;     // workspace of the fused path (the unfused buffers follow it)
  size_t off_gS = 0, off_gF = 0, off_gR = 0, off_gQ = 0;

  size_t state_elems() const { return (size_t)B * C * modes; }
  size_t src_bstride() const { return srcB > 1 ? (size_t)srcC * modes : 0; }
  size_t src_cstride() const { return srcC > 1 ? modes : 0; }
  size_t coef_bstride() const { return Bc > 1 ? (size_t)NCOEF * modes : 0; }
};

struct tfsm_graph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace {

template <class T>
int dev_alloc(tfsm_plan* p, T** ptr, size_t count, const char* what) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, count * sizeof(T) > 0 ? count * sizeof(T) : 16);
  if (e != hipSuccess) return hip_fail(e, what);
  p->allocs.push_back(q);
  *ptr = static_cast<T*>(q);
  return TFSM_OK;
}

// per-stage twiddle tables in the layout of Fft<N, VAR>::tw_offset: W^(r k), W = exp(-2 pi i/(Ns R))
template <int N, int VAR>
void twiddle_table_t(std::vector<float2>& h) {
  using F = Fft<N, VAR>;
  h.assign(F::tw_size(), make_float2(1.f, 0.f));
  for (int s = 1; s < F::NST; ++s) {
    const int R = F::radix(s), ns = F::ns_before(s), off = F::tw_offset(s);
    for (int r = 0; r < R; ++r)
      for (int k = 0; k < ns; ++k) {
        const double ang = -2.0 * M_PI * (double)r * (double)k / ((double)ns * R);
        h[off + r * ns + k] = make_float2((float)std::cos(ang), (float)std::sin(ang));
      }
  }
}

bool twiddle_table(int n, int var, std::vector<float2>& h) {
  if (var == 0) {
    switch (n) {
      case 16: twiddle_table_t<16, 0>(h); return true;
      case 32: twiddle_table_t<32, 0>(h); return true;
      case 64: twiddle_table_t<64, 0>(h); return true;
      case 128: twiddle_table_t<128, 0>(h); return true;
      case 256: twiddle_table_t<256, 0>(h); return true;
      case 512: twiddle_table_t<512, 0>(h); return true;
      case 1024: twiddle_table_t<1024, 0>(h); return true;
      case 2048: twiddle_table_t<2048, 0>(h); return true;
      case 4096: twiddle_table_t<4096, 0>(h); return true;
      case 48: twiddle_table_t<48, 0>(h); return true;
      case 96: twiddle_table_t<96, 0>(h); return true;
      case 100: twiddle_table_t<100, 0>(h); return true;
      case 112: twiddle_table_t<112, 0>(h); return true;
      case 192: twiddle_table_t<192, 0>(h); return true;
      case 200: twiddle_table_t<200, 0>(h); return true;
      case 384: twiddle_table_t<384, 0>(h); return true;
      case 400: twiddle_table_t<400, 0>(h); return true;
      case 768: twiddle_table_t<768, 0>(h); return true;
      case 800: twiddle_table_t<800, 0>(h); return true;
      default: return false;
    }
  }
  if (var == 2) {
    if (n == 128) {
      twiddle_table_t<128, 2>(h);
      return true;
    }
    return false;
  }
  if (var == 3) {
    switch (n) {
      case 16: twiddle_table_t<16, 3>(h); return true;
      case 32: twiddle_table_t<32, 3>(h); return true;
      case 64: twiddle_table_t<64, 3>(h); return true;
      case 128: twiddle_table_t<128, 3>(h); return true;
      case 256: twiddle_table_t<256, 3>(h); return true;
      default: return false;
    }
  }
  switch (n) {
    case 256: twiddle_table_t<256, 1>(h); return true;
    case 512: twiddle_table_t<512, 1>(h); return true;
    case 1024: twiddle_table_t<1024, 1>(h); return true;
    case 2048: twiddle_table_t<2048, 1>(h); return true;
    case 4096: twiddle_table_t<4096, 1>(h); return true;
    default: return false;
  }
}

int build_twiddles(tfsm_plan* p, int d) {
  for (int var = 0; var < 4; ++var) {
    std::vector<float2> h;
    if (!twiddle_table(p->n[d], var, h)) {
      p->tw[d][var] = nullptr;
      continue;
    }
    int rc = dev_alloc(p, &p->tw[d][var], h.size(), "twiddle table");
    if (rc) return rc;
    HIP_TRY(hipMemcpy(p->tw[d][var], h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload");
  }
  return TFSM_OK;
}

// tables of a long 1D mesh: stage twiddles of both factors and the four-step twiddles of the kept columns
int build_long1d(tfsm_plan* p) {
  const int len[2] = {p->l1, p->l2};
  float2** dst[2] = {&p->ltw1, &p->ltw2};
  for (int i = 0; i < 2; ++i) {
    std::vector<float2> h;
    if (!twiddle_table(len[i], long1d_var(len[i]), h)) return fail(TFSM_E_INVALID, "no radix plan for this length");
    int rc = dev_alloc(p, dst[i], h.size(), "twiddle table");
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*dst[i], h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload");
  }
  std::vector<float2> h((size_t)p->l1 * p->PF, make_float2(0.f, 0.f));
  for (int x1 = 0; x1 < p->l1; ++x1)
    for (int q2 = 0; q2 <= p->l2 / 2; ++q2) {
      const double ang = -2.0 * M_PI * (double)((long long)x1 * q2) / (double)p->n[0];
      h[(size_t)x1 * p->PF + q2] = make_float2((float)std::cos(ang), (float)std::sin(ang));
    }
  int rc = dev_alloc(p, &p->ltw4, h.size(), "four-step twiddles");
  if (rc) return rc;
  HIP_TRY(hipMemcpy(p->ltw4, h.data(), h.size() * sizeof(float2), hipMemcpyHostToDevice), "twiddle upload");
  return TFSM_OK;
}

// ---------------------------------------------------------------- transforms per axis
// Fixed-size kernels where the axis has them (rows: every length of the twiddle list; columns: up
// to 512 points), the general-length FFTs (gfft_run) elsewhere.
bool fast_rows(const tfsm_plan* p, int d) { return p->tw[d][0] != nullptr; }
bool fast_cols(const tfsm_plan* p, int d) { return p->tw[d][0] != nullptr && p->n[d] <= 512; }
bool axis_needs_gfft(const tfsm_plan* p, int d) { return d == p->D - 1 ? !fast_rows(p, d) : !fast_cols(p, d); }

// nrows rows of the last axis: GM_R2C (real in, ld in floats), GM_C2R, GM_C2C
hipError_t xf_rows(tfsm_plan* p, int mode, int dir, const void* in, size_t in_ld, void* out, size_t out_ld,
                   size_t nrows, float scale, hipStream_t st) {
  const int d = p->D - 1, n = p->n[d];
  if (nrows == 0) return hipSuccess;
  if (fast_rows(p, d) && nrows <= 0x7fffffffu) {
    if (mode == GM_R2C)
      return launch_rows_r2c(n, (const float*)in, in_ld, (float2*)out, out_ld, (int)nrows, scale, p->tw[d][0], st);
    if (mode == GM_C2R)
      return launch_rows_c2r(n, (const float2*)in, in_ld, (float*)out, out_ld, (int)nrows, scale, p->tw[d][0], st);
    return launch_rows_c2c(n, dir, (const float2*)in, in_ld, (float2*)out, out_ld, (int)nrows, scale, p->tw[d][0], st);
  }
  if (p->gax[d].n != n) return hipErrorInvalidValue;
  GLines li, lo;
  li.n_o = lo.n_o = nrows;
  li.os = in_ld;
  lo.os = out_ld;
  return gfft_run(p->gax[d], mode, dir, in, li, out, lo, scale, p->gtmp, st);
}

// complex transform along axis d < D - 1: nouter blocks of [n_d][...] with elements k * col_stride
// + i, i < ninner, of block o at o * outer_stride
hipError_t xf_cols(tfsm_plan* p, int d, int dir, const float2* in, float2* out, size_t nouter, size_t outer_stride,
                   size_t col_stride, size_t ninner, hipStream_t st) {
  if (nouter == 0 || ninner == 0) return hipSuccess;
  if (fast_cols(p, d) && ninner <= 0x7fffffffu)
    return launch_cols_c2c(p->n[d], dir, in, out, nouter, outer_stride, col_stride, (int)ninner, 1.0f, p->tw[d][0], st);
  if (p->gax[d].n != p->n[d]) return hipErrorInvalidValue;
  GLines l;
  l.n_o = nouter;
  l.n_i = ninner;
  l.os = outer_stride;
  l.is = 1;
  l.es = col_stride;
  return gfft_run(p->gax[d], GM_C2C, dir, in, l, out, l, 1.0f, p->gtmp, st);
}

// nblk real blocks [N0..N_{D-1}] -> half spectra [N0..][P]
int xf_forward_blocks(tfsm_plan* p, const float* u, float2* out, size_t nblk, hipStream_t st) {
  const int D = p->D, nl = p->n[D - 1];
  size_t rows = nblk;
  for (int d = 0; d < D - 1; ++d) rows *= p->n[d];
  HIP_TRY(xf_rows(p, GM_R2C, -1, u, (size_t)nl, out, (size_t)p->P, rows, 1.0f, st), "r2c launch");
  if (D == 2)
    HIP_TRY(xf_cols(p, 0, -1, out, out, nblk, p->modes, (size_t)p->P, (size_t)p->H, st), "column fft launch");
  if (D == 3) {
    const size_t plane = (size_t)p->n[1] * p->P;
    HIP_TRY(xf_cols(p, 1, -1, out, out, nblk * p->n[0], plane, (size_t)p->P, (size_t)p->H, st), "y fft launch");
    HIP_TRY(xf_cols(p, 0, -1, out, out, nblk, p->modes, plane, plane, st), "x fft launch");
  }
  return TFSM_OK;
}

// nblk half spectra -> real blocks, scaled by `scale`; `work` receives the partial transforms
// (it may be `in`, which is then overwritten; unused in 1D)
int xf_inverse_blocks(tfsm_plan* p, const float2* in, float2* work, float* u, size_t nblk, float scale,
                      hipStream_t st) {
  const int D = p->D, nl = p->n[D - 1];
  size_t rows = nblk;
  for (int d = 0; d < D - 1; ++d) rows *= p->n[d];
  if (D == 2) {
    HIP_TRY(xf_cols(p, 0, +1, in, work, nblk, p->modes, (size_t)p->P, (size_t)p->H, st), "column ifft launch");
    in = work;
  }
  if (D == 3) {
    const size_t plane = (size_t)p->n[1] * p->P;
    HIP_TRY(xf_cols(p, 0, +1, in, work, nblk, p->modes, plane, plane, st), "x ifft launch");
    HIP_TRY(xf_cols(p, 1, +1, work, work, nblk * p->n[0], plane, (size_t)p->P, (size_t)p->H, st), "y ifft launch");
    in = work;
  }
  HIP_TRY(xf_rows(p, GM_C2R, +1, in, (size_t)p->P, u, (size_t)nl, rows, scale, st), "c2r launch");
  return TFSM_OK;
}

// ---------------------------------------------------------------- unfused stepping
size_t plan_npts(const tfsm_plan* p) {
  size_t n = 1;
  for (int d = 0; d < p->D; ++d) n *= p->n[d];
  return n;
}

GenArgs gen_args(const tfsm_plan* p) {
  GenArgs g;
  g.term = p->term;
  g.D = p->D;
  g.B = p->B;
  g.C = p->C;
  for (int d = 0; d < 3; ++d) {
    g.n[d] = p->n[d];
    g.kmax[d] = p->kmax[d];
    g.kv[d] = p->kv[d];
  }
  g.H = p->H;
  g.P = p->P;
  g.modes = p->modes;
  g.npts = plan_npts(p);
  g.kv_bstride = p->kv_bstride;
  g.NF = gen_nf(p->term, p->C, p->D);
  g.NP = gen_np(p->term, p->C);
  g.coef_t = p->coef_t;
  return g;
}

// unfused buffers after the fused workspace: S (stage spectrum), F (fields, later product spectra),
// R (real fields), Q (real products)
void gen_layout(tfsm_plan* p) {
  if (p->genf) {
    p->ws_bytes = p->ws_fused;
    if (p->D == 2) {  // products and fields of the fused 2D layout
      p->off_P = roundup(p->ws_fused, 256);
      p->off_G = p->off_P + roundup(p->state_elems() * sizeof(float2), 256);
      p->ws_bytes = p->off_G + roundup((size_t)p->B * p->NF * p->n[0] * p->PF * sizeof(float2), 256);
    }
    return;
  }
  const GenArgs g = gen_args(p);
  const size_t sb = p->state_elems() * sizeof(float2);
  const size_t nfa = (size_t)(g.NF > g.NP ? g.NF : g.NP);
  p->off_gS = roundup(p->ws_fused, 256);
  p->off_gF = p->off_gS + roundup(sb, 256);
  p->off_gR = p->off_gF + roundup((size_t)p->B * nfa * p->modes * sizeof(float2), 256);
  p->off_gQ = p->off_gR + roundup((size_t)p->B * g.NF * g.npts * sizeof(float), 256);
  p->ws_bytes = p->off_gQ + roundup((size_t)p->B * g.NP * g.npts * sizeof(float), 256);
}

// general-length tables of the axes without fixed-size kernels, and their four-step scratch
int build_gaxes(tfsm_plan* p) {
  size_t tmp = 0;
  // blocks per transform: state channels, fields and products of both paths, adjoint fields
  int nb = p->C;
  const int counts[4] = {gen_nf(p->term, p->C, p->D), gen_np(p->term, p->C), 2 * p->C + p->C * p->D, 5};
  for (int c : counts) nb = c > nb ? c : nb;
  const size_t blk = (size_t)p->B * nb;
  for (int d = 0; d < p->D; ++d) {
    if (!axis_needs_gfft(p, d)) continue;
    hipError_t e = gaxis_build(p->gax[d], p->n[d], p->allocs);
    if (e == hipErrorInvalidValue) return fail(TFSM_E_INVALID, "mesh axis too long for the general-length FFT");
    HIP_TRY(e, "general FFT tables");
    // lines of one transform along axis d (full complex rows of tfsm_c2c included)
    size_t lines = blk;
    for (int e2 = 0; e2 < p->D - 1; ++e2)
      if (e2 != d) lines *= p->n[e2];
    if (d != p->D - 1) lines *= (size_t)p->n[p->D - 1] > (size_t)p->P ? (size_t)p->n[p->D - 1] : (size_t)p->P;
    const size_t t = gfft_tmp_elems(p->gax[d], lines);
    if (t > tmp) tmp = t;
  }
  if (tmp) return dev_alloc(p, &p->gtmp, tmp, "general FFT scratch");
  return TFSM_OK;
}

// Whether a general plan steps on the fused kernels of run-time lengths, and which axes take them (an axis
// with fixed-size kernels keeps those: they hold the transform in registers)
int plan_genfused(tfsm_plan* p) {
  if (p->cplx || p->force) return TFSM_OK;
  if (p->D == 1) {
    p->genf = p->genf_ok = (p->term == TERM_CONV || p->term == TERM_CONS) && p->C == 1 && genfused_mesh1d(p->gax[0]);
    return TFSM_OK;
  }
  if (p->D != 2 || p->term == TERM_CONS) return TFSM_OK;
  // fixed-size columns address whole pitch rows of the y wavenumber table (16 points at least); the paired
  // 512-point vorticity rows need an even number of rows per sample
  // where the rows are not of a fixed length: columns of 100, 112 and 200 points, whose fixed-size plans hold 16 and 20
  // values per thread (k2_col 112 points, 19 columns 28 us a launch), up to 1024 columns (vorticity SETDRK4 against the
  // unfused path, 112 points, B = 1, 4, 16, 64: fixed 0.97, 0.78, 0.62, 0.52, run-time 0.51, 0.42, 0.40, 0.44; Burgers
  // at B = 64 the reverse, 0.48, 0.48; an ETDRK2 step back, B = 1: 1.09, 0.74; 48, 96 and 192 points need no such rule)
  const bool slow_cols = (p->n[0] == 100 || p->n[0] == 112 || p->n[0] == 200) && (size_t)p->H * p->B <= 1024 &&
                         !row2d_supported(p->n[1], 0, 256);
  bool gen[2] = {!col2d_supported(p->n[0], 8, 0) || p->n[1] < 16 || slow_cols,
                 !row2d_supported(p->n[1], 0, 256) || (p->n[1] == 512 && p->n[0] % 2 != 0)};
  for (int d = 0; d < 2; ++d) {
    if (!gen[d]) continue;
    if (p->gax[d].n != p->n[d]) {
      hipError_t e = gaxis_build(p->gax[d], p->n[d], p->allocs);
      if (e != hipSuccess) return hip_fail(e, "general FFT tables");
    }
    if (!genfused_axis(p->gax[d])) return TFSM_OK;
  }
  // a few columns of over 2048 points of a two-channel product, whose six fields LDS holds one at a time: the unfused
  // launches spread them (2039 x 32, 8 SETDRK4 steps, us, unfused / fused: Burgers B = 1 3830 / 4256, B = 2 4157 / 4332,
  // B = 4 4756 / 4445; vorticity B = 1 3676 / 3383)
  const bool two = p->term == TERM_CONV || p->term == TERM_NSP;
  if (gen[0] && two && p->gax[0].g.L > 2048 && (size_t)p->H * p->B < 64) return TFSM_OK;
  p->genf = p->genf_ok = true;
  p->gf_col = gen[0];
  p->gf_row = gen[1];
  p->NF = p->term == TERM_KS ? 2 : 4;
  p->PF = (int)roundup((size_t)p->kmax[1] + 1, 16);
  return TFSM_OK;
}

// N(S) -> product spectra in F, and the batch mean of their DC for KSConvection; mask_in_place:
// S is zeroed outside the dealiasing box (the forced NSPressureConvection core does that)
int gen_eval(tfsm_plan* p, float2* S, char* ws, hipStream_t st, bool mask_in_place = false) {
  GenArgs g = gen_args(p);
  g.mask_in_place = mask_in_place ? 1 : 0;
  float2* F = (float2*)(ws + p->off_gF);
  float* R = (float*)(ws + p->off_gR);
  float* Q = (float*)(ws + p->off_gQ);
  HIP_TRY(launch_gen_fields(g, S, F, st), "field launch");
  int rc = xf_inverse_blocks(p, F, F, R, (size_t)p->B * g.NF, (float)(1.0 / (double)g.npts), st);
  if (rc) return rc;
  HIP_TRY(launch_gen_products(g, R, Q, st), "product launch");
  rc = xf_forward_blocks(p, Q, F, (size_t)p->B * g.NP, st);
  if (rc) return rc;
  if (p->ks_mean)
    HIP_TRY(launch_ks_dc(F, p->B, (size_t)g.NP * p->modes, 1, 0, (float2*)(ws + p->off_DC), st), "batch-mean launch");
  return TFSM_OK;
}

// evaluation from `in` and the stage combine `stage` (S receives the next stage spectrum).
// stepping: a forced NSPressureConvection masks the stage tensor it evaluates in place, as the
// reference's core does, except the state of a one-evaluation scheme, whose E u the reference
// forms before the evaluation (_etdrk.py:47-51, _setdrk_step.py:5-11)
int gen_stage(tfsm_plan* p, float2* in, float2* U, char* ws, int stage, StepMask m, hipStream_t st,
              bool stepping = false) {
  const bool forced = p->force != nullptr;
  int rc = gen_eval(p, in, ws, st, forced && stepping && stage != ST_R1_E0);
  if (rc) return rc;
  GenStageArgs s;
  s.stage = stage;
  s.Qs = (const float2*)(ws + p->off_gF);
  s.dc = p->ks_mean ? (const float2*)(ws + p->off_DC) : nullptr;
  s.U = U;
  s.A1 = (float2*)(ws + p->off_A1);
  s.A2 = (float2*)(ws + p->off_A2);
  s.S = (float2*)(ws + p->off_gS);
  s.coef = p->coef;
  s.coefc = p->cplx ? p->coefc : nullptr;
  s.coef_bstride = p->coef_bstride();
  s.coef_per_block = p->per_len ? 1 : 0;
  s.src = p->src;
  s.src_bstride = p->src_bstride();
  s.src_cstride = p->src_cstride();
  s.force = p->force;
  s.force_bstride = p->forceB > 1 ? (size_t)p->forceC * p->modes : 0;
  s.force_cstride = p->forceC > 1 ? p->modes : 0;
  s.masked_stage = forced && stepping ? 1 : 0;
  s.mask = m;
  HIP_TRY(launch_gen_stage(gen_args(p), s, st), "stage launch");
  return TFSM_OK;
}

int gen_step(tfsm_plan* p, float2* U, int nsteps, const int* rec_slot, void* traj, int T, char* ws, hipStream_t st,
             const int* act) {
  const int nev = scheme_evals(p->scheme);
  const size_t per = (size_t)p->C * p->modes;
  float2* S = (float2*)(ws + p->off_gS);
  StepMask m;
  m.act = act;
  int rc = TFSM_OK;
  for (int i = 0; i < nsteps && !rc; ++i) {
    m.it = i;
    if (rec_slot) rc = launch_status(launch_record(U, (float2*)traj, rec_slot, i, p->B, per, T, st), "record launch");
    for (int e = 0; e < nev && !rc; ++e)
      rc = gen_stage(p, e == 0 ? U : S, U, ws, scheme_stage(p->scheme, e), m, st, true);
  }
  if (rec_slot && !rc) rc = launch_status(launch_record(U, (float2*)traj, rec_slot, nsteps, p->B, per, T, st), "record launch");
  return rc;
}

int check_stream_errors(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, what);
  return TFSM_OK;
}

Row2Args row_args(tfsm_plan* p, char* ws, int b0, int nb) {
  Row2Args r;
  r.B = nb;
  r.N0 = p->n[0];
  r.N1 = p->n[1];
  r.H1 = p->H;
  r.P1 = p->P;
  r.PF = p->PF;
  r.kmax1 = p->kmax[1];
  r.NF = p->NF;
  r.tw1 = p->tw[1][plan2(p->n[1], p->row_var)];
  r.ay = p->kv[1];
  r.G = (const float2*)(ws + p->off_G);
  r.P = (float2*)(ws + p->off_P);
  r.b0 = b0;
  return r;
}

Col2Args col_args(tfsm_plan* p, float2* U, char* ws) {
  Col2Args c;
  c.B = p->B;
  c.C = p->C;
  c.N0 = p->n[0];
  c.N1 = p->n[1];
  c.H1 = p->H;
  c.P1 = p->P;
  c.PF = p->PF;
  c.kmax0 = p->kmax[0];
  c.kmax1 = p->kmax[1];
  c.NF = p->NF;
  c.coef_t = p->coef_t;
  c.scale = (float)(1.0 / ((double)p->n[0] * p->n[1]));
  c.tw0 = p->tw[0][plan2(p->n[0], p->col_var)];
  c.ax = p->kv[0];
  c.ay = p->kv[1];
  c.P = (const float2*)(ws + p->off_P);
  c.U = U;
  c.A1 = (float2*)(ws + p->off_A1);
  c.A2 = (float2*)(ws + p->off_A2);
  c.coef = p->coef;
  c.coef_bstride = p->coef_bstride();
  c.cpk = p->cpk;
  c.cpk_bstride = p->Bc > 1 ? 2 * p->modes : 0;
  c.c5t = p->c5t;
  c.ck01 = p->scheme == SETDRK4 ? p->ck01 : nullptr;
  c.c6t = p->scheme == SETDRK4 ? p->c6t : nullptr;
  c.src = p->src;
  c.src_bstride = p->src_bstride();
  c.src_cstride = p->src_cstride();
  c.src_cols = p->src_cols;
  if (p->src_bits_ok) {
    for (int w = 0; w < Col2Args::SRC_BIT_WORDS; ++w) c.src_bits[w] = p->src_bits[w];
    c.src_bits_ok = 1;
  }
  c.G = (float2*)(ws + p->off_G);
  c.dc = p->ks_mean ? (const float2*)(ws + p->off_DC) : nullptr;
  c.b0 = 0;
  c.nb = p->B;
  return c;
}

int launch_row(tfsm_plan* p, char* ws, int b0, int nb, hipStream_t st, StepMask m = StepMask()) {
  Row2Args r = row_args(p, ws, b0, nb);
  r.mask = m;
  if (p->gf_row) {
    HIP_TRY(launch_g2row(p->term, r, p->gax[1], st), "row kernel launch");
    return TFSM_OK;
  }
  HIP_TRY(launch_row2d(p->term, r, p->row_var, p->row_wg, st), "row kernel launch");
  return TFSM_OK;
}

int launch_col(tfsm_plan* p, float2* U, char* ws, int stage, int b0, int nb, hipStream_t st, StepMask m = StepMask()) {
  Col2Args c = col_args(p, U, ws);
  c.b0 = b0;
  c.mask = m;
  if (p->gf_col) {
    HIP_TRY(launch_g2col(p->term, c, p->gax[0], nb, stage, st), "column kernel launch");
    return TFSM_OK;
  }
  HIP_TRY(launch_col2d(p->term, c, nb, stage, p->V, p->col_var, st), "column kernel launch");
  return TFSM_OK;
}

// one nonlinear-evaluation pair of 2D kernels for samples [b0, b0 + nb)
int run2d_eval(tfsm_plan* p, float2* U, char* ws, int stage, int b0, int nb, hipStream_t st, StepMask m) {
  if (stage != ST_PRO) {
    int rc = launch_row(p, ws, b0, nb, st, m);
    if (rc) return rc;
    // KSConvection's mean couples the batch (the plan never splits it into sub-batches)
    if (p->ks_mean)
      HIP_TRY(launch_ks_dc((const float2*)(ws + p->off_P), p->B, p->modes, p->n[0], (size_t)p->P,
                           (float2*)(ws + p->off_DC), st),
              "batch-mean launch");
  }
  return launch_col(p, U, ws, stage, b0, nb, st, m);
}

// ---------------------------------------------------------------- 3D evaluation
Col3Args col3_args(tfsm_plan* p, float2* U, char* ws, int b0, int nb) {
  Col3Args c;
  c.B = p->B;
  c.N0 = p->n[0];
  c.N1 = p->n[1];
  c.N2 = p->n[2];
  c.H2 = p->H;
  c.P2 = p->P;
  c.PF2 = p->PF;
  c.K1 = p->K1;
  c.kmax0 = p->kmax[0];
  c.kmax1 = p->kmax[1];
  c.kmax2 = p->kmax[2];
  c.term = p->term;
  c.nc = p->C;
  c.coef_t = p->coef_t;
  c.scale = (float)(1.0 / ((double)p->n[0] * p->n[1] * p->n[2]));
  c.tw0 = p->tw[0][p->col_var == 1 ? 3 : var3(p->n[0])];
  c.ax = p->kv[0];
  c.ay = p->kv[1];
  c.az = p->kv[2];
  c.P = (const float2*)(ws + p->off_P);
  c.U = U;
  c.A1 = (float2*)(ws + p->off_A1);
  c.A2 = (float2*)(ws + p->off_A2);
  c.cpk = p->cpk;
  c.cpk_bstride = p->Bc > 1 ? 2 * p->modes : 0;
  c.c5t = p->c5t;
  c.ck01 = p->scheme == SETDRK4 ? p->ck01 : nullptr;
  c.c6t = p->scheme == SETDRK4 ? p->c6t : nullptr;
  c.src = p->src;
  c.src_bstride = p->src_bstride();
  c.src_cstride = p->src_cstride();
  c.G1 = (float2*)(ws + p->off_G);
  c.dc = p->ks_mean ? (const float2*)(ws + p->off_DC) : nullptr;
  c.b0 = b0;
  c.nb = nb;
  return c;
}

// one nonlinear evaluation of the 3D convection term for samples [b0, b0 + nb):
// z rows (products) -> y columns forward -> x columns (combine, fields) -> y columns inverse
// `parts` selects kernels (bit 0 z rows, 1 y forward, 2 x columns, 3 y inverse) for profiling.
int run3d_eval(tfsm_plan* p, float2* U, char* ws, int stage, int b0, int nb, hipStream_t st, int parts = 15,
               StepMask m = StepMask()) {
  const int N0 = p->n[0], N1 = p->n[1];
  float2* Pp = (float2*)(ws + p->off_P);
  if (stage != ST_PRO && (parts & 1)) {
    Row3Args r;
    r.term = p->term;
    r.N0 = N0;
    r.N1 = N1;
    r.N2 = p->n[2];
    r.P2 = p->P;
    r.PF2 = p->PF;
    r.kmax2 = p->kmax[2];
    r.tw2 = p->tw[2][p->row_var == 1 ? 3 : var3(p->n[2])];
    r.az = p->kv[2];
    r.G2 = (const float2*)(ws + p->off_G2);
    r.P = Pp;
    r.b0 = b0;
    r.nb = nb;
    r.mask = m;
    HIP_TRY(launch_row3d(r, p->row_var, st), "3D row kernel launch");
  }
  if (stage != ST_PRO && (parts & 2)) {
    float2* Pb = Pp + (size_t)b0 * p->C * p->modes;
    HIP_TRY(launch_cols_c2c(N1, -1, Pb, Pb, (size_t)nb * p->C * N0, (size_t)N1 * p->P, (size_t)p->P, p->H, 1.0f,
                            p->tw[1][0], st, m, b0, (size_t)p->C * N0),
            "3D y-forward launch");
    if (p->ks_mean)
      HIP_TRY(launch_ks_dc(Pp, p->B, p->modes, N0, (size_t)N1 * p->P, (float2*)(ws + p->off_DC), st),
              "batch-mean launch");
  }
  if (parts & 4) {
    Col3Args c = col3_args(p, U, ws, b0, nb);
    c.mask = m;
    HIP_TRY(launch_col3d(c, nb, stage, p->col_var, st), "3D column kernel launch");
  }
  if (!(parts & 8)) return TFSM_OK;
  Yinv3Args y;
  y.N0 = N0;
  y.N1 = N1;
  y.PF2 = p->PF;
  y.K1 = p->K1;
  y.kmax1 = p->kmax[1];
  y.kmax2 = p->kmax[2];
  y.nc = p->C;
  y.tw1 = p->tw[1][p->col_var == 1 ? 3 : var3(N1)];
  y.ay = p->kv[1];
  y.G1 = (const float2*)(ws + p->off_G);
  y.G2 = (float2*)(ws + p->off_G2);
  y.b0 = b0;
  y.nb = nb;
  y.mask = m;
  HIP_TRY(launch_yinv3d(y, p->col_var, st), "3D y-inverse launch");
  return TFSM_OK;
}

// one nonlinear evaluation of a long 1D mesh (row pass, then column pass with the stage combine)
int run_long1d(tfsm_plan* p, float2* U, char* ws, int stage, hipStream_t st) {
  Long1Args a;
  a.B = p->B * p->C;
  a.N = p->n[0];
  a.L1 = p->l1;
  a.L2 = p->l2;
  a.P = p->P;
  a.PG = p->PF;
  a.kmax = p->kmax[0];
  a.coef_t = p->coef_t;
  a.scale = (float)(1.0 / p->n[0]);
  a.tw1 = p->ltw1;
  a.tw2 = p->ltw2;
  a.tw4 = p->ltw4;
  a.ax = p->kv[0];
  a.ax_bstride = p->kv_bstride;
  a.U = U;
  a.A1 = (float2*)(ws + p->off_A1);
  a.A2 = (float2*)(ws + p->off_A2);
  a.cpk = p->cpk;
  a.cpk_bstride = p->Bc > 1 ? 2 * p->modes : 0;
  a.c5t = p->c5t;
  a.src = p->src;
  a.src_bstride = p->src_bstride();
  a.Pr = (const float2*)(ws + p->off_P);
  a.Pw = (float2*)(ws + p->off_P);
  a.G = (float2*)(ws + p->off_G);
  a.cons = p->term == TERM_CONS ? 1 : 0;
  if (stage != ST_PRO) HIP_TRY(launch_long1d_row(a, st), "1D row launch");
  HIP_TRY(launch_long1d_col(a, stage, st), "1D column launch");
  return TFSM_OK;
}

int run_eval(tfsm_plan* p, float2* U, char* ws, int stage, int b0, int nb, hipStream_t st, StepMask m = StepMask()) {
  return p->D == 3 ? run3d_eval(p, U, ws, stage, b0, nb, st, 15, m) : run2d_eval(p, U, ws, stage, b0, nb, st, m);
}

Run1Args run1_args(tfsm_plan* p, float2* U, char* ws) {
  Run1Args a;
  a.B = p->B * p->C;
  a.N = p->n[0];
  a.H = p->H;
  a.P = p->P;
  a.kmax = p->kmax[0];
  a.coef_t = p->coef_t;
  a.scale = (float)(1.0 / p->n[0]);
  a.scheme = p->scheme;
  a.tw = p->tw[0][0];
  a.tw_run = p->tw[0][var1(p->n[0])];
  a.ax = p->kv[0];
  a.ax_bstride = p->kv_bstride;
  a.U = U;
  a.A1 = (float2*)(ws + p->off_A1);
  a.A2 = (float2*)(ws + p->off_A2);
  a.coef = p->coef;
  a.coef_bstride = p->coef_bstride();
  a.coefc = p->cplx ? p->coefc : nullptr;
  a.cpk = p->cpk;
  a.cpk_bstride = p->Bc > 1 ? 2 * p->modes : 0;
  a.cons = p->term == TERM_CONS ? 1 : 0;
  a.src = p->src;
  a.src_bstride = p->src_bstride();
  a.nsteps = 0;
  a.nsteps_per = nullptr;
  a.rec_slot = nullptr;
  a.traj = nullptr;
  a.T = 0;
  a.eval_only = 0;
  return a;
}

hipError_t run1d(tfsm_plan* p, const Run1Args& a, hipStream_t st) {
  return p->genf ? launch_g1run(a, p->gax[0], st) : launch_run1d(a, st);
}

// act: optional per-sample step counts (device int32 [B], 2D / 3D): sample b advances by
// min(act[b], nsteps) steps and is not touched after that
int step_impl(tfsm_plan* p, void* uh, int nsteps, const int* rec_slot, void* traj, int T, void* ws, hipStream_t st,
              const int* act = nullptr) {
  float2* U = (float2*)uh;
  if (p->scheme == ETDRK0) {
    if (p->cplx)
      HIP_TRY(launch_linear_steps_c(U, p->coefc + CS_E * p->modes, p->coef_bstride(), p->modes, p->C,
                                    p->state_elems(), nsteps, rec_slot, (float2*)traj, T, st),
              "linear step launch");
    else
      HIP_TRY(launch_linear_steps(U, p->coef + CS_E * p->modes, p->coef_bstride(), p->modes, p->C, p->state_elems(),
                                  nsteps, rec_slot, (float2*)traj, T, st),
              "linear step launch");
    return TFSM_OK;
  }
  if (!ws) return fail(TFSM_E_INVALID, "workspace pointer is null");
  if (p->general && !p->genf) return gen_step(p, U, nsteps, rec_slot, traj, T, (char*)ws, st, act);
  if (p->D == 1 && p->term == TERM_KS) {
    // one launch per stage (the batch mean couples the samples): raw product -> mean -> combine
    Run1Args a = run1_args(p, U, (char*)ws);
    float2* S = (float2*)((char*)ws + p->off_S);
    float2* Nr = (float2*)((char*)ws + p->off_N);
    float2* dc = p->ks_mean ? (float2*)((char*)ws + p->off_DC) : nullptr;
    const int nev = scheme_evals(p->scheme);
    const size_t per = (size_t)p->C * p->modes;
    for (int i = 0; i < nsteps; ++i) {
      if (rec_slot) HIP_TRY(launch_record(U, (float2*)traj, rec_slot, i, p->B, per, T, st), "record launch");
      for (int e = 0; e < nev; ++e) {
        HIP_TRY(launch_k1_eval_ks(a, e == 0 ? U : S, Nr, st), "1D product launch");
        if (dc) HIP_TRY(launch_ks_dc(Nr, a.B, (size_t)p->P, 1, 0, dc, st), "batch-mean launch");
        HIP_TRY(launch_k1_stage(a, scheme_stage(p->scheme, e), Nr, dc, S, st), "1D stage launch");
      }
    }
    if (rec_slot) HIP_TRY(launch_record(U, (float2*)traj, rec_slot, nsteps, p->B, per, T, st), "record launch");
    return TFSM_OK;
  }
  if (p->D == 1 && p->l1) {
    const int nev = scheme_evals(p->scheme);
    const size_t per = (size_t)p->C * p->modes;
    if (int rc = run_long1d(p, U, (char*)ws, ST_PRO, st)) return rc;
    for (int i = 0; i < nsteps; ++i) {
      if (rec_slot) HIP_TRY(launch_record(U, (float2*)traj, rec_slot, i, p->B, per, T, st), "record launch");
      for (int e = 0; e < nev; ++e)
        if (int rc = run_long1d(p, U, (char*)ws, scheme_stage(p->scheme, e), st)) return rc;
    }
    if (rec_slot) HIP_TRY(launch_record(U, (float2*)traj, rec_slot, nsteps, p->B, per, T, st), "record launch");
    return TFSM_OK;
  }
  if (p->D == 1) {
    Run1Args a = run1_args(p, U, (char*)ws);
    a.nsteps = nsteps;
    a.rec_slot = rec_slot;
    a.traj = (float2*)traj;
    a.T = T;
    HIP_TRY(run1d(p, a, st), "1D stepper launch");
    return TFSM_OK;
  }
  if (p->D == 2 && p->persistent && run2d_supported(p->term, p->n[0], p->n[1], p->PF) && !p->cplx) {
    // one workgroup per sample runs every step (small meshes: launch-bound otherwise)
    Col2Args ca = col_args(p, U, (char*)ws);
    Row2Args ra = row_args(p, (char*)ws, 0, p->B);
    // k2_run has a radix plan of its own, whatever the tiled kernels' tuning
    ca.tw0 = p->tw[0][RUN2D_VAR];
    ra.tw1 = p->tw[1][RUN2D_VAR];
    Run2Args r;
    r.b0 = 0;
    r.nb = p->B;
    r.scheme = p->scheme;
    r.nsteps = nsteps;
    r.act = act;
    r.rec_slot = rec_slot;
    r.traj = (float2*)traj;
    r.T = T;
    r.per_sample = (size_t)p->C * p->modes;
    HIP_TRY(launch_run2d(p->term, ca, ra, r, st), "persistent 2D stepper launch");
    return TFSM_OK;
  }
  if (p->D >= 2) {
    // Temporal blocking: a sub-batch of samples goes through many steps before the next one, so
    // its state, auxiliary stages, products and fields stay resident in the last-level cache
    // across the 2 * evals launches of every step.  Samples are independent: same results.
    // With several streams, sub-batch k runs on stream k % ns (fork from and join back into the
    // caller's stream with events, which also holds under graph capture): their kernels overlap
    // and fill each other's latency.  Sub-batches use disjoint parts of the workspace.
    const int nev = scheme_evals(p->scheme);
    const int sb = (p->sub_batch > 0 && p->sub_batch < p->B) ? p->sub_batch : p->B;
    const size_t per = (size_t)p->C * p->modes;
    // streams in use: no more than there are sub-batches
    const int nsub = (p->B + sb - 1) / sb;
    const int ns = p->nstreams < nsub ? p->nstreams : nsub;
    if (ns > 1) {
      HIP_TRY(hipEventRecord(p->ev_fork, st), "fork event");
      for (int i = 0; i + 1 < ns; ++i) HIP_TRY(hipStreamWaitEvent(p->aux[i], p->ev_fork, 0), "fork wait");
    }
    // On several streams the steps are queued in rounds (every sub-batch gets its next steps
    // before the following round starts): a stream's hardware queue holds a bounded number of
    // packets and the host blocks once one is full, so queuing all steps of one sub-batch first
    // would leave the other streams idle until that sub-batch is nearly done.  A first round of
    // one step starts every stream early.  One stream: a single round, every step of a
    // sub-batch before the next.
    const int round0 = ns > 1 ? 1 : nsteps, round = ns > 1 ? 16 : nsteps;
    const hipStream_t caller = st;
    int rc = TFSM_OK;
    for (int s0 = 0, r = 0; !rc; ++r) {
      const int len = r == 0 ? round0 : round;
      const int s1 = nsteps - s0 < len ? nsteps : s0 + len;
      for (int b0 = 0, k = 0; b0 < p->B && !rc; b0 += sb, ++k) {
        st = (k % ns) ? p->aux[k % ns - 1] : caller;
        const int nb = (p->B - b0) < sb ? (p->B - b0) : sb;
        float2* Ub = U + (size_t)b0 * per;
        float2* Tb = traj ? (float2*)traj + (size_t)b0 * T * per : nullptr;
        StepMask m;
        m.act = act;
        m.it = s0;
        if (s0 == 0) rc = run_eval(p, U, (char*)ws, ST_PRO, b0, nb, st, m);
        for (int i = s0; i < s1 && !rc; ++i) {
          m.it = i;
          if (rec_slot) rc = launch_status(launch_record(Ub, Tb, rec_slot, i, nb, per, T, st), "record launch");
          for (int e = 0; e < nev && !rc; ++e)
            rc = run_eval(p, U, (char*)ws, scheme_stage(p->scheme, e), b0, nb, st, m);
        }
        if (s1 == nsteps && rec_slot && !rc)
          rc = launch_status(launch_record(Ub, Tb, rec_slot, nsteps, nb, per, T, st), "record launch");
      }
      if (s1 == nsteps) break;
      s0 = s1;
    }
    // the joins are recorded on every exit, also after a failed launch: work already queued on the
    // auxiliary streams is then still ordered before anything the caller queues next
    for (int i = 0; i + 1 < ns; ++i) {
      const int jr = launch_status(hipEventRecord(p->ev_join[i], p->aux[i]), "join event");
      const int jw = jr ? jr : launch_status(hipStreamWaitEvent(caller, p->ev_join[i], 0), "join wait");
      if (!rc) rc = jw;
    }
    return rc;
  }
  return fail(TFSM_E_INVALID, "stepping is not available for this dimension");
}

// ---------------------------------------------------------------- adjoint helpers
AdjArgs adj_args(tfsm_plan* p) {
  AdjArgs a;
  a.D = p->D;
  a.C = p->C;
  a.B = p->B;
  a.npts = 1;
  for (int d = 0; d < 3; ++d) {
    a.n[d] = p->n[d];
    a.kmax[d] = p->kmax[d];
    a.kv[d] = p->kv[d];
    if (d < p->D) a.npts *= p->n[d];
  }
  a.H = p->H;
  a.P = p->P;
  a.modes = p->modes;
  a.coef_t = p->coef_t;
  a.term = p->term;
  return a;
}

struct AdjLayout {
  size_t Aa, N0s, T1, Jv, Ab, Nb, Na, Ac, Nc, Cb, Bb, Abar, part, F, Fs, X, Q;
  size_t Ga, Gb, Gc, Qs, GP;  // fused 2D path
  size_t total;
};

// fields and products of the transposed Jacobian (k_adj_fields / k_adj_products)
int adj_nfa(const tfsm_plan* p) { return p->term == TERM_VC ? 5 : 2 * p->C + p->C * p->D; }
int adj_nq(const tfsm_plan* p) { return p->term == TERM_VC ? 4 : p->C + p->C * p->D; }

// 2D plans of the fused kernels whose axes k_adjoint2d.hip covers
bool adj_fused(const tfsm_plan* p) {
  return p->D == 2 && p->fused_ok && !p->general && adj2d_size(p->n[0]) && adj2d_size(p->n[1]) && !p->force &&
         (p->term == TERM_VC ? p->C == 1 : p->term == TERM_CONV && p->C == 2);
}

// workgroups per sample of the coefficient gradient: 512 modes each, up to 256
int adj_grad_blocks(const tfsm_plan* p) {
  const size_t n = ((size_t)p->C * p->modes + 511) / 512;
  return n > 256 ? 256 : (int)n;
}

AdjLayout adj_layout(const tfsm_plan* p) {
  const int nfa = adj_nfa(p), nq = adj_nq(p);
  size_t npts = 1;
  for (int d = 0; d < p->D; ++d) npts *= p->n[d];
  const size_t S = roundup(p->state_elems() * sizeof(float2), 256);
  const bool four = p->scheme == SETDRK4;
  AdjLayout l = {};
  size_t o = 0;
  auto take = [&](size_t& at, size_t bytes) { at = o; o += roundup(bytes, 256); };
  take(l.part, (size_t)p->B * adj_grad_blocks(p) * sizeof(double));
  take(l.Na, S);
  take(l.Ab, S);
  if (four) {
    take(l.Nb, S);
    take(l.Nc, S);
    take(l.Cb, S);
    take(l.Bb, S);
  }
  if (adj_fused(p)) {
    const size_t fields = (size_t)p->B * 4 * p->n[0] * p->PF * sizeof(float2);
    take(l.Ga, fields);
    if (four) {
      take(l.Gb, fields);
      take(l.Gc, fields);
    }
    take(l.Qs, fields);
    take(l.GP, S);
    l.total = o;
    return l;
  }
  take(l.Aa, S);
  take(l.N0s, S);
  take(l.T1, S);
  take(l.Jv, S);
  if (!four) take(l.Nb, S);
  if (four) {
    take(l.Ac, S);
    take(l.Abar, S);
  }
  take(l.F, (size_t)p->B * nfa * p->modes * sizeof(float2));
  take(l.Fs, (size_t)p->B * (nfa > nq ? nfa : nq) * p->modes * sizeof(float2));
  take(l.X, (size_t)p->B * nfa * npts * sizeof(float));
  take(l.Q, (size_t)p->B * nq * npts * sizeof(float));
  l.total = o;
  return l;
}

// W = J_N(U)^T V (Convection, 1D / 2D)
int adj_jt(tfsm_plan* p, const float2* U, const float2* V, float2* W, char* wsa, hipStream_t st) {
  const AdjLayout l = adj_layout(p);
  const AdjArgs a = adj_args(p);
  const int nfa = adj_nfa(p), nq = adj_nq(p);
  float2* F = (float2*)(wsa + l.F);
  float2* Fs = (float2*)(wsa + l.Fs);
  float* X = (float*)(wsa + l.X);
  float* Q = (float*)(wsa + l.Q);
  HIP_TRY(launch_adj_fields(a, U, V, F, st), "adjoint fields launch");
  const float scale = (float)(1.0 / (double)a.npts);
  int rc = xf_inverse_blocks(p, F, Fs, X, (size_t)p->B * nfa, scale, st);
  if (rc) return rc;
  HIP_TRY(launch_adj_products(a, X, Q, st), "adjoint products launch");
  rc = xf_forward_blocks(p, Q, Fs, (size_t)p->B * nq, st);
  if (rc) return rc;
  HIP_TRY(launch_adj_combine(a, Fs, W, st), "adjoint combine launch");
  return TFSM_OK;
}

// N(U) -> workspace A1
int eval_nonlinear(tfsm_plan* p, float2* U, char* ws, hipStream_t st) {
  if (p->general && !p->genf) return gen_stage(p, U, U, ws, ST_EVAL, StepMask(), st);
  if (p->l1 && !p->general) {
    int rc = run_long1d(p, U, ws, ST_PRO, st);
    return rc ? rc : run_long1d(p, U, ws, ST_EVAL, st);
  }
  if (p->D == 1) {
    Run1Args r = run1_args(p, U, ws);
    r.eval_only = 1;
    r.nsteps = 1;
    HIP_TRY(run1d(p, r, st), "1D evaluation launch");
    return TFSM_OK;
  }
  int rc = run_eval(p, U, ws, ST_PRO, 0, p->B, st);
  if (!rc) rc = run_eval(p, U, ws, ST_EVAL, 0, p->B, st);
  return rc;
}

AdjLinArgs lin_args(tfsm_plan* p, float2* Y) {
  AdjLinArgs a;
  a.B = p->B;
  a.C = p->C;
  a.P = p->P;
  a.H = p->H;
  a.modes = p->modes;
  a.coef = p->coef;
  a.coef_bstride = p->coef_bstride();
  a.nt = 0;
  a.Y = Y;
  return a;
}

void lin_term(AdjLinArgs& a, const float2* X, int slot, float s) {
  a.X[a.nt] = X;
  a.slot[a.nt] = slot;
  a.s[a.nt] = s;
  ++a.nt;
}

AdjGradArgs grad_args(tfsm_plan* p, char* wsa, double* grad) {
  AdjGradArgs g;
  g.B = p->B;
  g.C = p->C;
  g.P = p->P;
  g.H = p->H;
  g.nlast = p->n[p->D - 1];
  g.modes = p->modes;
  g.coef = p->coef;
  g.coef_bstride = p->coef_bstride();
  g.dcoef = p->dcoef;
  g.dcoef_bstride = p->Bc > 1 ? (size_t)ADJ_NDCOEF * p->modes : 0;
  g.sym = p->sym;
  g.nt = 0;
  g.nblk = adj_grad_blocks(p);
  g.part = (double*)(wsa + adj_layout(p).part);
  g.out = grad;
  return g;
}

// one term s dc c <X, Y>
void grad_term(AdjGradArgs& g, const float2* X, const float2* Y, int dslot, float s, int cslot = -1) {
  g.X[g.nt] = X;
  g.Y[g.nt] = Y;
  g.dslot[g.nt] = dslot;
  g.cslot[g.nt] = cslot;
  g.s[g.nt++] = s;
}

enum { D_E = 0, D_C1 = 1, D_C2 = 2 };                                                // slots of 1- and 2-stage schemes
enum { D4_E = 0, D4_E2 = 1, D4_C1 = 2, D4_C4 = 3, D4_C5 = 4, D4_C6 = 5 };  // of SETDRK4

// SETDRK4's coefficient gradient; a = E2 u + c1 N0 enters as its two terms
int adj_grad4(tfsm_plan* p, const float2* U, const float2* Ubn, const float2* N0, const float2* Na, const float2* Nb,
              const float2* Nc, const float2* Cb, const float2* Bb, const float2* Ab, char* wsa, double* grad,
              hipStream_t st) {
  AdjGradArgs g = grad_args(p, wsa, grad);
  grad_term(g, Ubn, U, D4_E, 1.f);
  grad_term(g, Ubn, N0, D4_C4, 1.f);
  grad_term(g, Ubn, Na, D4_C5, 2.f);
  grad_term(g, Ubn, Nb, D4_C5, 2.f);
  grad_term(g, Ubn, Nc, D4_C6, 1.f);
  grad_term(g, Cb, U, D4_E2, 1.f, CS_E2);
  grad_term(g, Cb, N0, D4_E2, 1.f, CS_C1);
  grad_term(g, Cb, Nb, D4_C1, 2.f);
  grad_term(g, Cb, N0, D4_C1, -1.f);
  grad_term(g, Bb, U, D4_E2, 1.f);
  grad_term(g, Bb, Na, D4_C1, 1.f);
  grad_term(g, Ab, U, D4_E2, 1.f);
  grad_term(g, Ab, N0, D4_C1, 1.f);
  HIP_TRY(launch_adj_grad(g, st), "adjoint gradient launch");
  return TFSM_OK;
}

// One adjoint step on the fused kernels (k_adjoint2d.hip).  The step's own stages run on k2_row and k2_col
// into one field array each; on the way back, every stage is a row launch (products, and with `grad` that
// state's own product) and a column launch that ends in the next stage's adjoint fields.
int adj_step_fused(tfsm_plan* p, float2* U, const float2* Ubn, float2* Ubo, double* grad, char* W, char* A,
                   hipStream_t st) {
  const AdjLayout l = adj_layout(p);
  const bool want = grad && p->adj_term >= 0;
  float2* Pr = (float2*)(W + p->off_P);
  float2* A1 = (float2*)(W + p->off_A1);  // N0
  float2* Gu = (float2*)(W + p->off_G);
  float2 *Ga = (float2*)(A + l.Ga), *Gb = (float2*)(A + l.Gb), *Gc = (float2*)(A + l.Gc);
  float2 *Na = (float2*)(A + l.Na), *Nb = (float2*)(A + l.Nb), *Nc = (float2*)(A + l.Nc);
  float2 *Ab = (float2*)(A + l.Ab), *Bb = (float2*)(A + l.Bb), *Cb = (float2*)(A + l.Cb);
  Adj2RowArgs r;
  r.B = p->B;
  r.N0 = p->n[0];
  r.N1 = p->n[1];
  r.P1 = p->P;
  r.PF = p->PF;
  r.kmax1 = p->kmax[1];
  r.tw1 = p->tw[1][adj2d_var(p->n[1])];
  r.ay = p->kv[1];
  r.GP = (float2*)(A + l.GP);
  r.Q = (float2*)(A + l.Qs);
  Adj2ColArgs base;
  base.B = p->B;
  base.N0 = p->n[0];
  base.H1 = p->H;
  base.P1 = p->P;
  base.PF = p->PF;
  base.kmax0 = p->kmax[0];
  base.kmax1 = p->kmax[1];
  base.coef_t = p->coef_t;
  base.scale = (float)(1.0 / ((double)p->n[0] * p->n[1]));
  base.tw0 = p->tw[0][adj2d_var(p->n[0])];
  base.ax = p->kv[0];
  base.ay = p->kv[1];
  base.coef = p->coef;
  base.coef_bstride = p->coef_bstride();
  base.P = Pr;
  base.src = p->src;
  base.src_bstride = p->src_bstride();
  base.src_cstride = p->src_cstride();
  base.Q = nullptr;
  base.N = base.Y = base.GP = nullptr;
  base.nt = base.nv = 0;
  base.yslot = CS_C1;
  base.ys = 0.f;
  auto x_term = [](Adj2ColArgs& c, const float2* X, int slot, float s) {
    c.X[c.nt] = X;
    c.slot[c.nt] = slot;
    c.s[c.nt++] = s;
  };
  auto v_term = [](Adj2ColArgs& c, const float2* X, int slot, float s) {
    c.V[c.nv] = X;
    c.vslot[c.nv] = slot;
    c.vs[c.nv++] = s;
  };
  // fields of stage `stage`'s result into G (the last array the stage reads is the product in ws)
  auto stage = [&](int sc, float2* G) -> int {
    Col2Args c = col_args(p, U, W);
    c.G = G;
    HIP_TRY(launch_col2d(p->term, c, p->B, sc, p->V, p->col_var, st), "column kernel launch");
    return TFSM_OK;
  };
  auto rows = [&](float2* G) -> int {
    Row2Args q = row_args(p, W, 0, p->B);
    q.G = G;
    HIP_TRY(launch_row2d(p->term, q, p->row_var, p->row_wg, st), "row kernel launch");
    return TFSM_OK;
  };
  auto in = [&](int slot) -> int {  // c u'bar -> GP
    Adj2ColArgs c = base;
    v_term(c, Ubn, slot, 1.f);
    c.GP = (float2*)(A + l.GP);
    HIP_TRY(launch_adj2d_col(p->term, c, st), "adjoint column launch");
    return TFSM_OK;
  };
  // products of the fields G with the adjoint fields, then the column pass c; N(state) -> N with `want`
  auto back = [&](Adj2ColArgs& c, const float2* G, float2* N) -> int {
    r.G = G;
    r.P = want && N ? Pr : nullptr;
    HIP_TRY(launch_adj2d_row(p->term, r, st), "adjoint row launch");
    c.Q = r.Q;
    c.N = want ? N : nullptr;
    HIP_TRY(launch_adj2d_col(p->term, c, st), "adjoint column launch");
    return TFSM_OK;
  };
  int rc = stage(ST_PRO, Gu);
  if (rc) return rc;
  if (p->scheme == SETDRK4) {
    if ((rc = rows(Gu)) || (rc = stage(ST_R4_E0, Ga)) || (rc = rows(Ga)) || (rc = stage(ST_R4_E1, Gb)) ||
        (rc = rows(Gb)) || (rc = stage(ST_R4_E2, Gc)) || (rc = in(CS_C6)))
      return rc;
    Adj2ColArgs c = base;  // cbar = J(c)^T c6 u'bar;  Nb bar = 2 c1 cbar + 2 c5 u'bar
    c.Y = Cb;
    c.ys = 2.f;
    v_term(c, Ubn, CS_C5, 2.f);
    c.GP = (float2*)(A + l.GP);
    if ((rc = back(c, Gc, Nc))) return rc;
    c = base;  // bbar = J(b)^T Nb bar;  Na bar = c1 bbar + 2 c5 u'bar
    c.Y = Bb;
    c.ys = 1.f;
    v_term(c, Ubn, CS_C5, 2.f);
    c.GP = (float2*)(A + l.GP);
    if ((rc = back(c, Gb, Nb))) return rc;
    c = base;  // abar = E2 cbar + J(a)^T Na bar;  N0 bar = c1 abar - c1 cbar + c4 u'bar
    x_term(c, Cb, CS_E2, 1.f);
    c.Y = Ab;
    c.ys = 1.f;
    v_term(c, Cb, CS_C1, -1.f);
    v_term(c, Ubn, CS_C4, 1.f);
    c.GP = (float2*)(A + l.GP);
    if ((rc = back(c, Ga, Na))) return rc;
    c = base;  // ubar = E u'bar + E2 bbar + E2 abar + J(u)^T N0 bar
    x_term(c, Ubn, CS_E, 1.f);
    x_term(c, Bb, CS_E2, 1.f);
    x_term(c, Ab, CS_E2, 1.f);
    c.Y = Ubo;
    if ((rc = back(c, Gu, nullptr))) return rc;
    return want ? adj_grad4(p, U, Ubn, A1, Na, Nb, Nc, Cb, Bb, Ab, A, grad, st) : TFSM_OK;
  }
  const bool two = p->scheme == ETDRK2 || p->scheme == SETDRK2;
  AdjGradArgs g = grad_args(p, A, grad);
  if (two) {
    if ((rc = rows(Gu)) || (rc = stage(scheme_stage(p->scheme, 0), Ga)) || (rc = in(CS_C2))) return rc;
    Adj2ColArgs c = base;  // abar = u'bar + J(a)^T c2 u'bar;  N0 bar = c1 abar - c2 u'bar
    x_term(c, Ubn, -1, 1.f);
    c.Y = Ab;
    c.ys = 1.f;
    v_term(c, Ubn, CS_C2, -1.f);
    c.GP = (float2*)(A + l.GP);
    if ((rc = back(c, Ga, Na))) return rc;
    c = base;  // ubar = E abar + J(u)^T N0 bar
    x_term(c, Ab, CS_E, 1.f);
    c.Y = Ubo;
    if ((rc = back(c, Gu, nullptr))) return rc;
    grad_term(g, Ubn, Na, D_C2, 1.f);
    grad_term(g, Ubn, A1, D_C2, -1.f);
    grad_term(g, Ab, U, D_E, 1.f);
    grad_term(g, Ab, A1, D_C1, 1.f);
  } else {
    if ((rc = in(CS_C1))) return rc;
    Adj2ColArgs c = base;  // ubar = E u'bar + J(u)^T c1 u'bar
    x_term(c, Ubn, CS_E, 1.f);
    c.Y = Ubo;
    if ((rc = back(c, Gu, Na))) return rc;  // (Na: N0 here)
    grad_term(g, Ubn, U, D_E, 1.f);
    grad_term(g, Ubn, Na, D_C1, 1.f);
  }
  if (want) HIP_TRY(launch_adj_grad(g, st), "adjoint gradient launch");
  return TFSM_OK;
}

// One adjoint SETDRK4 step (see k_adjoint.hip): recompute N0, a, Na, b, Nb, c (and Nc for the
// coefficient gradient) from u, then the transposed stages from c back to u.
int adjoint_step4(tfsm_plan* p, float2* U, const float2* Ubn, float2* Ubo, double* grad, char* W, char* A,
                  hipStream_t st) {
  const AdjLayout l = adj_layout(p);
  float2* A1 = (float2*)(W + p->off_A1);
  float2* N0 = (float2*)(A + l.N0s);
  float2* Sa = (float2*)(A + l.Aa);
  float2* Na = (float2*)(A + l.Na);
  float2* Sb = (float2*)(A + l.Ab);
  float2* Nb = (float2*)(A + l.Nb);
  float2* Sc = (float2*)(A + l.Ac);
  float2* Nc = (float2*)(A + l.Nc);
  float2* T = (float2*)(A + l.T1);
  float2* Jv = (float2*)(A + l.Jv);
  float2* Cb = (float2*)(A + l.Cb);
  float2* Bb = (float2*)(A + l.Bb);
  float2* Ab = (float2*)(A + l.Abar);
  const bool want = grad && p->adj_term >= 0;
  const size_t sbytes = p->state_elems() * sizeof(float2);
  auto nonlin = [&](float2* X, float2* out) -> int {
    int rc = eval_nonlinear(p, X, W, st);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(out, A1, sbytes, hipMemcpyDeviceToDevice, st), "adjoint copy");
    return TFSM_OK;
  };
  auto comb = [&](AdjLinArgs& a) -> int {
    HIP_TRY(launch_adj_lincomb(a, st), "adjoint stage launch");
    return TFSM_OK;
  };
  int rc = nonlin(U, N0);
  if (rc) return rc;
  AdjLinArgs a = lin_args(p, Sa);  // a = E2 u + c1 N0
  lin_term(a, U, CS_E2, 1.f);
  lin_term(a, N0, CS_C1, 1.f);
  if ((rc = comb(a)) || (rc = nonlin(Sa, Na))) return rc;
  a = lin_args(p, Sb);  // b = E2 u + c1 Na
  lin_term(a, U, CS_E2, 1.f);
  lin_term(a, Na, CS_C1, 1.f);
  if ((rc = comb(a)) || (rc = nonlin(Sb, Nb))) return rc;
  a = lin_args(p, Sc);  // c = E2 a + c1 (2 Nb - N0)
  lin_term(a, Sa, CS_E2, 1.f);
  lin_term(a, Nb, CS_C1, 2.f);
  lin_term(a, N0, CS_C1, -1.f);
  if ((rc = comb(a))) return rc;
  if (want && (rc = nonlin(Sc, Nc))) return rc;
  // backward
  a = lin_args(p, T);  // Nc bar = c6 u'bar
  lin_term(a, Ubn, CS_C6, 1.f);
  if ((rc = comb(a)) || (rc = adj_jt(p, Sc, T, Cb, A, st))) return rc;
  a = lin_args(p, T);  // Nb bar = 2 c5 u'bar + 2 c1 cbar
  lin_term(a, Ubn, CS_C5, 2.f);
  lin_term(a, Cb, CS_C1, 2.f);
  if ((rc = comb(a)) || (rc = adj_jt(p, Sb, T, Bb, A, st))) return rc;
  a = lin_args(p, T);  // Na bar = 2 c5 u'bar + c1 bbar
  lin_term(a, Ubn, CS_C5, 2.f);
  lin_term(a, Bb, CS_C1, 1.f);
  if ((rc = comb(a)) || (rc = adj_jt(p, Sa, T, Jv, A, st))) return rc;
  a = lin_args(p, Ab);  // abar = E2 cbar + J(a)^T Na bar
  lin_term(a, Cb, CS_E2, 1.f);
  lin_term(a, Jv, -1, 1.f);
  if ((rc = comb(a))) return rc;
  a = lin_args(p, T);  // N0 bar = c4 u'bar - c1 cbar + c1 abar
  lin_term(a, Ubn, CS_C4, 1.f);
  lin_term(a, Cb, CS_C1, -1.f);
  lin_term(a, Ab, CS_C1, 1.f);
  if ((rc = comb(a)) || (rc = adj_jt(p, U, T, Jv, A, st))) return rc;
  a = lin_args(p, Ubo);  // ubar = E u'bar + E2 bbar + E2 abar + J(u)^T N0 bar
  lin_term(a, Ubn, CS_E, 1.f);
  lin_term(a, Bb, CS_E2, 1.f);
  lin_term(a, Ab, CS_E2, 1.f);
  lin_term(a, Jv, -1, 1.f);
  if ((rc = comb(a))) return rc;
  return want ? adj_grad4(p, U, Ubn, N0, Na, Nb, Nc, Cb, Bb, Ab, A, grad, st) : TFSM_OK;
}

AdjStageArgs stage_args(tfsm_plan* p, int op) {
  AdjStageArgs s;
  s.op = op;
  s.two_stage = (p->scheme == ETDRK2 || p->scheme == SETDRK2) ? 1 : 0;
  s.B = p->B;
  s.C = p->C;
  s.P = p->P;
  s.H = p->H;
  s.modes = p->modes;
  s.coef = p->coef;
  s.coef_bstride = p->coef_bstride();
  s.X0 = s.X1 = nullptr;
  s.Y0 = s.Y1 = nullptr;
  return s;
}

}  // namespace

// Device address of `scratch` on device `dev`, resolved once per device with that device current.
static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

static int scratch_on_device(int dev, void** out) {
  if (dev < 0 || dev >= kMaxDevices) return fail(TFSM_E_INVALID, "device index out of range for the static scratch");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* q = nullptr;
    const hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "address of the static scratch");
    if (!q) return fail(TFSM_E_DEVICE, "address of the static scratch is null");
    g_scratch_ptr[dev] = q;
  }
  *out = g_scratch_ptr[dev];
  return TFSM_OK;
}

// nbatch blocks of the plan's [C][N...] shape: at least one, and few enough that every launch's row
// count fits the kernels' 32-bit row index
static int check_nbatch(const tfsm_plan* p, int32_t nbatch) {
  if (nbatch < 1) return fail(TFSM_E_INVALID, "nbatch must be >= 1");
  size_t rows = (size_t)nbatch * p->C;
  for (int d = 0; d < p->D - 1; ++d) rows *= p->n[d];
  if (rows * p->n[p->D - 1] > (size_t)INT32_MAX) return fail(TFSM_E_INVALID, "nbatch too large for one call");
  return TFSM_OK;
}

extern "C" {

const char* tfsm_last_error(void) { return g_err.c_str(); }

int tfsm_version(void) { return (0 << 16) | 1; }

int tfsm_plan_create(const tfsm_geometry* geom, const tfsm_terms* terms, void* stream, tfsm_plan** out) {
  if (!geom || !terms || !out) return fail(TFSM_E_INVALID, "null argument");
  *out = nullptr;
  const int D = geom->ndim;
  if (D < 1 || D > 3) return fail(TFSM_E_INVALID, "the engine supports 1D, 2D and 3D meshes");
  if (geom->batch < 1 || geom->channels < 1) return fail(TFSM_E_INVALID, "batch and channels must be >= 1");
  // sizes the fused kernels cover; any other size (>= 2 points per axis) runs the unfused path
  bool fused_sizes = true;
  for (int d = 0; d < D; ++d) {
    if (!(geom->length[d] > 0)) return fail(TFSM_E_INVALID, "mesh lengths must be positive");
    const int n = geom->n[d];
    if (n < 2) return fail(TFSM_E_INVALID, "mesh axes need at least 2 points");
    const bool ok = D == 1   ? ((is_pow2(n) && n >= 32 && n <= 4096) || is_mixed_size(n))
                    : D == 2 ? ((is_pow2(n) && n >= 16 && n <= 1024) || is_mixed_size_2d(n))
                             : ((is_pow2(n) && n >= 16 && n <= 256) || is_mixed_size_3d(n));
    fused_sizes = fused_sizes && ok;
  }
  const bool ks_keep = terms->nonlinear == TFSM_TERM_KS_KEEP_MEAN;
  const int term = ks_keep ? TERM_KS : terms->nonlinear;
  if (term != TERM_NONE && term != TERM_CONV && term != TERM_VC && term != TERM_NSP && term != TERM_KS &&
      term != TERM_CONS)
    return fail(TFSM_E_INVALID, "unknown nonlinear term");
  if (term == TERM_CONS && geom->channels != D)
    return fail(TFSM_E_INVALID, "convection operator only works for vector field with the same dimension as mesh");
  if (term == TERM_KS && geom->channels != 1) return fail(TFSM_E_INVALID, "KSConvection only supports scalar field");
  if ((term == TERM_CONV || term == TERM_NSP) && geom->channels != D)
    return fail(TFSM_E_INVALID, "convection operator only works for vector field with the same dimension as mesh");
  if (term == TERM_NSP && D == 1)
    return fail(TFSM_E_INVALID, "term not supported by engine: NSPressureConvection on a 1D mesh");
  if (term == TERM_VC && (D != 2 || geom->channels != 1))
    return fail(TFSM_E_INVALID, "Only vorticity in 2Dmesh is supported");
  if (terms->n_linear < 0 || terms->n_linear > 4) return fail(TFSM_E_INVALID, "at most 4 linear terms");
  bool cplx = false;
  for (int t = 0; t < terms->n_linear; ++t) {
    const int kind = terms->linear_kind[t];
    if (kind < TFSM_LIN_LAP || kind > TFSM_LIN_DERIV) return fail(TFSM_E_INVALID, "unknown linear term");
    if (kind != TFSM_LIN_DERIV) continue;
    if (terms->linear_dim[t] < 0 || terms->linear_dim[t] >= D)
      return fail(TFSM_E_INVALID, "SpatialDerivative axis out of range");
    if (terms->linear_order[t] < 1 || terms->linear_order[t] > 8)
      return fail(TFSM_E_INVALID, "SpatialDerivative order must be 1..8");
    if (geom->channels != 1) return fail(TFSM_E_INVALID, "The SpatialDerivative operator only supports scalar field.");
    if (terms->linear_order[t] & 1) cplx = true;
  }
  // the fused kernels cover every product term on their sizes, except ConservativeConvection in 3D
  // and a complex L with a product term in 2D / 3D; the unfused path covers the rest
  bool fused = fused_sizes && !(term == TERM_CONS && D == 3) && !(cplx && term != TERM_NONE && D > 1);
  if (fused && D == 3 && term != TERM_NONE && term != TERM_CONS)
    fused = step3d_supported(geom->n[0], geom->n[1], geom->n[2]);
  // long 1D meshes that split into two fixed-size lengths (k_long1d.hip)
  int l1 = 0, l2 = 0;
  if (D == 1 && !fused_sizes && !cplx && geom->channels == 1 && (term == TERM_CONV || term == TERM_CONS) &&
      geom->n[0] > 4096 && long1d_split(geom->n[0], &l1, &l2))
    fused = true;
  if (terms->n_linear > 0 && !terms->linear_coef) return fail(TFSM_E_INVALID, "linear coefficients missing");
  const int Bc = terms->coef_batch < 1 ? 1 : terms->coef_batch;
  if (Bc != 1 && Bc != geom->batch) return fail(TFSM_E_INVALID, "coef_batch must be 1 or the batch size");
  if (geom->length_per_sample && D != 1) return fail(TFSM_E_INVALID, "per-sample lengths are 1D only");

  hipStream_t st = (hipStream_t)stream;
  int device = 0;
  HIP_TRY(hipGetDevice(&device), "current device");
  tfsm_plan* p = new tfsm_plan();
  p->device = device;
  p->D = D;
  p->B = geom->batch;
  p->C = geom->channels;
  for (int d = 0; d < D; ++d) {
    p->n[d] = geom->n[d];
    p->len[d] = geom->length[d];
  }
  p->H = p->n[D - 1] / 2 + 1;
  p->P = (int)roundup(p->H, 16);
  p->modes = (size_t)p->P;
  for (int d = 0; d < D - 1; ++d) p->modes *= p->n[d];
  p->term = term;
  p->ks_mean = term == TERM_KS && !ks_keep;
  p->coef_t = terms->nonlinear_coef;
  p->rate = terms->dealias_rate > 0 ? terms->dealias_rate : 2.0 / 3.0;
  p->nlin = terms->n_linear;
  for (int t = 0; t < p->nlin; ++t) {
    p->lin_kind[t] = terms->linear_kind[t];
    // the axis and order fields are read only for the terms that have them
    if (p->lin_kind[t] == TFSM_LIN_DERIV) {
      p->lin_dim[t] = terms->linear_dim[t];
      p->lin_order[t] = terms->linear_order[t];
    }
  }
  p->cplx = cplx;
  p->fused_ok = fused;
  p->general = !fused && term != TERM_NONE;
  p->l1 = l1;
  p->l2 = l2;
  p->per_len = D == 1 && geom->length_per_sample;
  p->Bc = Bc;
  int rc = TFSM_OK;
  for (int d = 0; d < D; ++d) {
    p->kmax[d] = dealias_kmax(p->n[d], p->len[d], p->rate);
    if (p->kmax[d] < -1) {
      tfsm_plan_destroy(p);
      return fail(TFSM_E_INVALID, "dealias mask is not an index range");
    }
    rc = build_twiddles(p, d);
    if (rc) break;
  }
  if (!rc) rc = build_gaxes(p);
  if (!rc && p->l1) {
    p->PF = (int)roundup((size_t)p->l2 / 2 + 1, 16);
    rc = build_long1d(p);
  }
  // axis wavenumber tables
  if (!rc) {
    for (int d = 0; d < D && !rc; ++d) {
      if (D == 1 && geom->length_per_sample) {
        std::vector<float> all((size_t)p->B * p->C * p->n[0]), a;
        for (int b = 0; b < p->B; ++b) {
          axis_table(p->n[0], geom->length_per_sample[b], a);
          for (int c = 0; c < p->C; ++c)
            std::memcpy(&all[((size_t)b * p->C + c) * p->n[0]], a.data(), a.size() * sizeof(float));
        }
        rc = dev_alloc(p, &p->kv[0], all.size(), "axis table");
        if (!rc) {
          hipError_t e = hipMemcpy(p->kv[0], all.data(), all.size() * sizeof(float), hipMemcpyHostToDevice);
          if (e != hipSuccess) rc = hip_fail(e, "axis table upload");
        }
        p->kv_bstride = (size_t)p->n[0];
      } else {
        std::vector<float> a;
        axis_table(p->n[d], p->len[d], a);
        rc = dev_alloc(p, &p->kv[d], a.size(), "axis table");
        if (!rc) {
          hipError_t e = hipMemcpy(p->kv[d], a.data(), a.size() * sizeof(float), hipMemcpyHostToDevice);
          if (e != hipSuccess) rc = hip_fail(e, "axis table upload");
        }
      }
    }
  }
  // linear symbol L per (coefficient sample, mode)
  const int Lb = (D == 1 && geom->length_per_sample) ? p->B * p->C : Bc;
  if (D == 1 && geom->length_per_sample) p->Bc = Lb;
  if (!rc) rc = dev_alloc(p, &p->L, (size_t)Lb * p->modes, "linear symbol");
  if (!rc) rc = dev_alloc(p, &p->coef, (size_t)Lb * NCOEF * p->modes, "coefficient table");
  if (!rc) rc = dev_alloc(p, &p->cpk, (size_t)Lb * 2 * p->modes, "packed coefficient table");
  if (!rc) rc = dev_alloc(p, &p->c5t, (size_t)Lb * p->modes, "c5 table");
  if (!rc) rc = dev_alloc(p, &p->ck01, (size_t)Lb * p->modes, "SETDRK4 [E2, c1] table");
  if (!rc) rc = dev_alloc(p, &p->c6t, (size_t)Lb * p->modes, "SETDRK4 c6 table");
  if (!rc && cplx) rc = dev_alloc(p, &p->Lc, (size_t)Lb * p->modes, "complex linear symbol");
  if (!rc && cplx) rc = dev_alloc(p, &p->coefc, (size_t)Lb * NCOEF * p->modes, "complex coefficient table");
  if (!rc) {
    hipError_t e = hipMemsetAsync(p->coef, 0, (size_t)Lb * NCOEF * p->modes * sizeof(float), st);
    if (e != hipSuccess) rc = hip_fail(e, "coefficient table clear");
  }
  if (!rc) {
    LinArgs la;
    la.D = D;
    for (int d = 0; d < 3; ++d) {
      la.n[d] = p->n[d];
      la.kv[d] = p->kv[d];
    }
    la.H = p->H;
    la.P = p->P;
    la.modes = p->modes;
    la.kv_bstride = p->kv_bstride;
    la.nterm = p->nlin;
    for (int t = 0; t < 4; ++t) {
      la.kind[t] = t < p->nlin ? terms->linear_kind[t] : 0;
      la.dim[t] = p->lin_dim[t];
      la.order[t] = p->lin_order[t];
    }
    la.Bc = Lb;
    la.L = p->L;
    la.Lc = p->Lc;
    float* dcoef = nullptr;
    std::vector<float> hc((size_t)(p->nlin > 0 ? p->nlin : 1) * Lb, 0.f);
    for (int t = 0; t < p->nlin; ++t)
      for (int b = 0; b < Lb; ++b) {
        const int src_b = (Bc == 1) ? 0 : (D == 1 && geom->length_per_sample ? b / p->C : b);
        hc[(size_t)t * Lb + b] = terms->linear_coef[(size_t)t * Bc + src_b];
      }
    rc = dev_alloc(p, &dcoef, hc.size(), "linear coefficients");
    if (!rc) {
      hipError_t e = hipMemcpy(dcoef, hc.data(), hc.size() * sizeof(float), hipMemcpyHostToDevice);
      if (e != hipSuccess) rc = hip_fail(e, "linear coefficient upload");
    }
    la.coef = dcoef;
    for (int t = 0; t < 4; ++t) la.cval[t] = 0.f;
    if (!rc) {
      hipError_t e = launch_linear_symbol(la, st);
      if (e != hipSuccess) rc = hip_fail(e, "linear symbol launch");
    }
  }
  // workspace layout
  if (!rc) {
    const size_t sb = p->state_elems() * sizeof(float2);
    p->off_A1 = 0;
    p->off_A2 = roundup(sb, 256);
    if (!p->fused_ok) {
      p->ws_bytes = p->off_A2 + roundup(sb, 256);
    } else if (D == 3) {
      // products P [B][3][N0][N1][P2]; fields G1 [B][6][N0][K1][PF2]; G2 [B][9][N0][N1][PF2]
      p->PF = (int)roundup((size_t)p->kmax[2] + 1, 16);
      p->K1 = 2 * p->kmax[1] + 1;
      p->off_P = p->off_A2 + roundup(sb, 256);
      p->off_G = p->off_P + roundup(sb, 256);
      p->off_G2 = p->off_G + roundup((size_t)p->B * 6 * p->n[0] * p->K1 * p->PF * sizeof(float2), 256);
      p->ws_bytes = p->off_G2 + roundup((size_t)p->B * 9 * p->n[0] * p->n[1] * p->PF * sizeof(float2), 256);
    } else if (D == 2) {
      p->NF = (term == TERM_KS || term == TERM_CONS) ? 2 : 4;
      p->PF = (int)roundup((size_t)p->kmax[1] + 1, 16);
      p->off_P = p->off_A2 + roundup(sb, 256);
      // ConservativeConvection keeps two product planes per channel
      p->off_G = p->off_P + roundup(term == TERM_CONS ? 2 * sb : sb, 256);
      p->ws_bytes = p->off_G + roundup((size_t)p->B * p->NF * p->n[0] * p->PF * sizeof(float2), 256);
    } else if (p->l1) {
      const size_t plane = (size_t)p->B * p->l1 * p->PF * sizeof(float2);
      p->off_P = p->off_A2 + roundup(sb, 256);
      p->off_G = p->off_P + roundup(plane, 256);
      p->ws_bytes = p->off_G + roundup((term == TERM_CONS ? 1 : 2) * plane, 256);
    } else {
      p->ws_bytes = p->off_A2 + roundup(sb, 256);
      if (term == TERM_KS) {
        p->off_S = p->ws_bytes;
        p->off_N = p->off_S + roundup(sb, 256);
        p->ws_bytes = p->off_N + roundup(sb, 256);
      }
    }
    p->off_DC = p->ws_bytes;
    p->ws_bytes += 256;
    p->ws_fused = p->ws_bytes;
    if (p->general) rc = plan_genfused(p);
    if (!rc && p->general) gen_layout(p);
  }
  // default launch shape (the autotuner may refine it)
  if (!rc && D == 2 && (p->fused_ok || p->genf)) {
    const int n0 = p->n[0], n1 = p->n[1];
    // measured per axis size: 512 keeps 16-column tiles; 64, 128 and 256 run 8-column tiles and rows of 4
    // values per thread.  Their launches are one round of workgroups, as long as one thread's chain of
    // transforms, and shorter chains win at every batch (SETDRK4, us per step, against the plans of 8 and
    // 16 values per thread that these replace: Burgers 128^2 B = 1 141 -> 62, B = 16 133 -> 70, B = 64 195
    // -> 111; vorticity 64^2 B = 4 54 -> 42, 128^2 B = 16 97 -> 58, 256^2 B = 8 95 -> 80, B = 32 136 -> 122)
    if (n0 == 64 || n0 == 128 || n0 == 256) {
      p->V = 8;
      p->col_var = 1;
    }
    // 1024-point columns: 8 columns per tile (LDS), the 8-values-per-thread plan (the 16-value
    // plan holds 2 waves per SIMD and spills for NSPressureConvection and ConservativeConvection)
    if (n0 == 1024) {
      p->V = 8;
      p->col_var = 1;
    }
    if (n1 == 64 || n1 == 128 || n1 == 256) {
      p->row_var = 1;
      // few rows: one-wavefront workgroups spread over more CUs (128^2 B = 1 63.9 -> 61.5; B = 16 the reverse)
      if ((size_t)p->B * n0 <= 512) p->row_wg = 64;
    }
    // Sub-batches of about 2M points on two streams, from 2M points per batch: the tail of one sub-batch's
    // launch overlaps the other's next pass and its arrays stay in the cache.  On one stream they only
    // shorten the launches (SETDRK4, us per step, one stream / whole batch / two streams: vorticity 128^2
    // B = 256 382 / 184 / 157, 100^2 B = 256 401 / 229 / 228; Burgers 128^2 B = 256 378 / 263 / 221;
    // NavierStokes 256^2 B = 64 338 / 286 / 255).  Other lines where sweeps drew them:
    const bool pair = term == TERM_CONV || term == TERM_NSP, one = term == TERM_VC || term == TERM_KS;
    const int B = p->B;
    const size_t pt = (size_t)n0 * n1, pts = (size_t)B * pt, sub_pts = (size_t)1 << 21;
    int sub = 0, ns = 2;
    if (pts >= sub_pts) {
      const int parts = pts / sub_pts > 2 ? (int)(pts / sub_pts) : 2;
      sub = (B + parts - 1) / parts;
    }
    // samples of `of` points in all, and no split below two such sub-batches
    auto of_points = [&](size_t of, int least) {
      const int lim = (int)(of / pt) > least ? (int)(of / pt) : least;
      return B >= 2 * lim ? lim : 0;
    };
    // 512-point columns.  One channel: 4M points, 16 samples at least (vorticity 512^2 B = 64 614 us, 721 by 2M and
    // 717 whole; 512 x 64 B = 64 136 whole, 151 in halves; 512 x 128 B = 256 661, 705 by 2M).  Two channels on
    // rows of 512 points or more: 16 samples from B = 32 (Burgers 512^2 505 us, 555 by 2M; 512 x 256 the reverse)
    if (n0 == 512 && one) sub = of_points((size_t)1 << 22, 16);
    if (n0 == 512 && pair && n1 >= 512 && B >= 32) sub = 16;
    // 1024-point columns.  Two channels on rows of 512 points or more: 4M points (Burgers 1024^2 B = 8 650 us, 840
    // by 2M; 1024 x 512 B = 16 594, 651 by 2M; 1024 x 256 B = 64 1264 by 2M, 1312).  One channel: 4M points on
    // shorter rows, 8M on these (vorticity 1024 x 256 B = 64 835 us, 920 whole; 1024^2 B = 16 875, 894 whole,
    // 1085 by 4M)
    if (n0 == 1024 && pair && n1 >= 512) sub = of_points((size_t)1 << 22, 1);
    if (n0 == 1024 && one) sub = of_points((size_t)1 << (n1 < 512 ? 22 : 23), 1);
    // ConservativeConvection on long columns: from 4M points (512^2 B = 32 547 us, 714 whole; at 2M points 1024 x 256
    // B = 8 256, 243 whole; 256 x 1024 B = 8 202, 190; 128 x 1024 B = 16 the reverse, 154, 161)
    if (n0 >= 256 && term == TERM_CONS && pts < 2 * sub_pts) sub = 0;
    // KSConvection, with two fields instead of four: from 4M points (256 x 1024 B = 8, 2M points: 123 us, 112 whole;
    // 128^2 B = 128 104, 93; at 4M points 135, 143 whole)
    if (term == TERM_KS && pts < 2 * sub_pts) sub = 0;
    // 256^2 up to 95 samples: 16 samples on two streams, on four from B = 48 (Burgers B = 48: 233 -> 180 us)
    if (n0 == 256 && n1 == 256 && term != TERM_NSP && p->B >= (term == TERM_KS ? 64 : 32) && p->B < 96) {
      sub = 16;
      ns = p->B >= 48 ? 4 : 2;
    }
    // (a plan without a product term steps in one elementwise launch)
    if (sub > 0 && sub < p->B && !p->ks_mean && !p->genf && term != TERM_NONE) {
      p->sub_batch = sub;
      rc = tfsm_plan_set_streams(p, ns);
    }
    // 512-point two-channel columns: 8 columns per tile where a launch has few tiles (Burgers B = 16 in
    // sub-batches of 8, 4 values more per thread: 272 -> 236 us; NavierStokes, every batch: B = 4 138 -> 128,
    // B = 32 596 -> 578)
    if (n0 == 512 && (term == TERM_NSP || (term == TERM_CONV && p->B >= 16 && p->B < 32))) {
      p->V = 8;
      p->col_var = term == TERM_CONV ? 1 : 0;
    }
  }
  // small square meshes step with the persistent per-sample kernel (one launch per call)
  if (!rc && D == 2 && p->fused_ok && run2d_supported(term, p->n[0], p->n[1], p->PF) && !p->cplx)
    p->persistent = true;
  // 3D plans of 4 values per thread: z rows from 32 points; the columns of meshes up to 32 points along x and y,
  // and up to 64 for NSPressureConvection (with its stage kernels), whose launches are as long as one thread's
  // chain of transforms (SETDRK4, us per step: NSP 64^3 B = 2 224 -> 180, B = 16 947 -> 778, 32^3 B = 4 197 ->
  // 130; Burgers 32^3 B = 4 194 -> 140; at 64^3 Burgers, and at 128 points, no gain)
  if (!rc && D == 3 && is_pow2(p->n[0]) && is_pow2(p->n[1]) && is_pow2(p->n[2])) {
    const int nxy = p->n[0] > p->n[1] ? p->n[0] : p->n[1];
    p->row_var = p->n[2] >= 32 ? 1 : 0;
    p->col_var = nxy == 32 || (nxy == 64 && term == TERM_NSP) ? 1 : 0;
  }
  // 3D Convection and NSPressureConvection: sub-batches on several streams, so that one's VALU-bound z-row pass
  // overlaps another's memory-bound column passes and their launches' tails (whole batch -> sub-batches, us
  // per step).  Meshes of 800k points or more: one sample each on two streams (96^3 B = 4 NavierStokes 1248
  // -> 1052, 100^3 B = 2 1304 -> 935, 128^3 B = 2 Burgers ETDRK2 363 -> 331), pairs at 128^3 from B = 4.
  // Smaller ones, down to 100k points, from 800k points per batch: two halves (48^3 B = 8 NavierStokes 410 ->
  // 296, 64^3 B = 4 247 -> 239; 32^3 loses at every batch), pairs on four streams at 64^3 from B = 8.
  const bool conv3 = D == 3 && p->fused_ok && (term == TERM_CONV || term == TERM_NSP);
  if (!rc && conv3 && p->B >= 2) {
    const size_t npts = (size_t)p->n[0] * p->n[1] * p->n[2], pts = npts * p->B;
    int sub = 0, ns = 2;
    if (npts >= 800000) sub = 1;
    else if (npts >= 100000 && pts >= 800000) sub = (p->B + 1) / 2;
    if (p->n[0] == 128 && p->n[1] == 128 && p->n[2] == 128 && p->B >= 4) sub = 2;
    if (p->n[0] == 64 && p->n[1] == 64 && p->n[2] == 64 && p->B >= 8) {
      sub = 2;
      ns = 4;
    }
    if (sub > 0) {
      p->sub_batch = sub;
      rc = tfsm_plan_set_streams(p, ns);
    }
  }
  if (rc) {
    tfsm_plan_destroy(p);
    return rc;
  }
  *out = p;
  return TFSM_OK;
}

int tfsm_plan_destroy(tfsm_plan* plan) {
  if (!plan) return TFSM_OK;
  for (int i = 0; i + 1 < TFSM_MAX_STREAMS; ++i) {
    if (plan->aux[i]) {
      (void)hipStreamSynchronize(plan->aux[i]);
      (void)hipStreamDestroy(plan->aux[i]);
    }
    if (plan->ev_join[i]) (void)hipEventDestroy(plan->ev_join[i]);
  }
  if (plan->ev_fork) (void)hipEventDestroy(plan->ev_fork);
  for (void* q : plan->allocs) (void)hipFree(q);
  delete plan;
  return TFSM_OK;
}

int64_t tfsm_plan_pitch(const tfsm_plan* plan) { return plan ? plan->P : 0; }

int64_t tfsm_plan_state_elems(const tfsm_plan* plan) { return plan ? (int64_t)plan->state_elems() : 0; }

int64_t tfsm_plan_workspace_bytes(const tfsm_plan* plan) { return plan ? (int64_t)plan->ws_bytes : 0; }

int64_t tfsm_plan_inverse_scratch_bytes(const tfsm_plan* plan, int32_t nbatch) {
  if (!plan) return 0;
  if (plan->D == 1) return 0;
  return (int64_t)((size_t)nbatch * plan->C * plan->modes * sizeof(float2));
}

int tfsm_plan_set_tuning(tfsm_plan* plan, int32_t col_tile, int32_t col_var, int32_t row_var, int32_t row_wg,
                         int32_t sub_batch) {
  if (!plan) return fail(TFSM_E_INVALID, "null plan");
  if (plan->l1) return fail(TFSM_E_INVALID, "the kernels of long 1D meshes have no launch shape");
  if (!plan->fused_ok) return fail(TFSM_E_INVALID, "no fixed-size fused kernels for this plan: it has no launch shape");
  if (plan->D == 3 && (row_var < 0 || row_var > 1 || col_var < 0 || col_var > 1))
    return fail(TFSM_E_INVALID, "unsupported 3D tuning");
  if (plan->D == 3 && (col_var == 1 || row_var == 1) &&
      (!is_pow2(plan->n[0]) || !is_pow2(plan->n[1]) || !is_pow2(plan->n[2])))
    return fail(TFSM_E_INVALID, "the radix-4 3D plans need power-of-two axes");
  if (plan->D == 2) {
    if (!col2d_supported(plan->n[0], col_tile, col_var)) return fail(TFSM_E_INVALID, "unsupported column tuning");
    if ((plan->P % col_tile) != 0) return fail(TFSM_E_INVALID, "column tile must divide the pitch");
    if (!row2d_supported(plan->n[1], row_var, row_wg)) return fail(TFSM_E_INVALID, "unsupported row tuning");
  }
  if (sub_batch > 0 && sub_batch < plan->B && plan->ks_mean)
    return fail(TFSM_E_INVALID, "KSConvection couples the batch through its mean: no sub-batches");
  plan->V = col_tile;
  plan->col_var = col_var;
  plan->row_var = row_var;
  plan->row_wg = row_wg;
  plan->sub_batch = sub_batch < 0 ? 0 : sub_batch;
  return TFSM_OK;
}

int tfsm_plan_get_tuning(const tfsm_plan* plan, int32_t* out) {
  if (!plan || !out) return fail(TFSM_E_INVALID, "null argument");
  out[0] = plan->V;
  out[1] = plan->col_var;
  out[2] = plan->row_var;
  out[3] = plan->row_wg;
  out[4] = plan->sub_batch;
  out[5] = plan->nstreams;
  return TFSM_OK;
}

int tfsm_plan_set_persistent(tfsm_plan* plan, int32_t on) {
  if (!plan) return fail(TFSM_E_INVALID, "null plan");
  if (on && plan->general) return fail(TFSM_E_INVALID, "the plan has no fixed-size fused kernels, or set_general(1)");
  if (on && !(plan->D == 2 && run2d_supported(plan->term, plan->n[0], plan->n[1], plan->PF) && !plan->cplx))
    return fail(TFSM_E_INVALID, "the persistent 2D stepper covers square 32^2 and 64^2 meshes with Convection or "
                                "VorticityConvection (2/3 dealiasing or coarser)");
  plan->persistent = on != 0;
  return TFSM_OK;
}

int32_t tfsm_plan_persistent(const tfsm_plan* plan) { return plan && plan->persistent ? 1 : 0; }

int tfsm_plan_set_general(tfsm_plan* plan, int32_t on) {
  if (!plan) return fail(TFSM_E_INVALID, "null plan");
  if (on) {
    if (plan->term == TERM_NONE) return fail(TFSM_E_INVALID, "a plan without a product term has no nonlinear evaluation");
    plan->general = true;
    plan->genf = false;
    plan->persistent = false;
    gen_layout(plan);
    return TFSM_OK;
  }
  if (plan->genf_ok) {
    plan->genf = true;
    gen_layout(plan);
    return TFSM_OK;
  }
  if (!plan->fused_ok) return fail(TFSM_E_INVALID, "no fused kernels for this plan: it steps through the unfused path");
  plan->general = false;
  plan->ws_bytes = plan->ws_fused;
  return TFSM_OK;
}

int32_t tfsm_plan_general(const tfsm_plan* plan) { return plan && plan->general ? 1 : 0; }

int32_t tfsm_plan_path(const tfsm_plan* plan) {
  if (!plan || plan->term == TERM_NONE) return TFSM_PATH_LINEAR;
  if (plan->general) return plan->genf ? TFSM_PATH_RUNTIME : TFSM_PATH_UNFUSED;
  return plan->l1 ? TFSM_PATH_LONG1D : TFSM_PATH_FIXED;
}

int tfsm_plan_set_streams(tfsm_plan* plan, int32_t nstreams) {
  if (!plan) return fail(TFSM_E_INVALID, "null plan");
  if (nstreams < 1 || nstreams > TFSM_MAX_STREAMS) return fail(TFSM_E_INVALID, "nstreams must be 1 to 4");
  if (nstreams > 1 && plan->ks_mean)
    return fail(TFSM_E_INVALID, "KSConvection couples the batch through its mean: one stream only");
  if (nstreams > 1 && !plan->ev_fork)
    HIP_TRY(hipEventCreateWithFlags(&plan->ev_fork, hipEventDisableTiming), "fork event");
  for (int i = 0; i + 1 < nstreams; ++i) {
    if (plan->aux[i]) continue;
    // default priority, non-blocking with respect to the null stream
    HIP_TRY(hipStreamCreateWithFlags(&plan->aux[i], hipStreamNonBlocking), "auxiliary stream");
    HIP_TRY(hipEventCreateWithFlags(&plan->ev_join[i], hipEventDisableTiming), "join event");
  }
  plan->nstreams = nstreams;
  return TFSM_OK;
}

int tfsm_plan_set_scheme(tfsm_plan* plan, int32_t scheme, double dt, int32_t n_points, double radius, void* stream) {
  if (!plan) return fail(TFSM_E_INVALID, "null plan");
  if (scheme < ETDRK0 || scheme > SETDRK4) return fail(TFSM_E_INVALID, "unknown scheme");
  const bool nonlinear = plan->term != TERM_NONE || plan->src != nullptr;
  if (scheme == ETDRK0 && nonlinear) return fail(TFSM_E_INVALID, "The ETDRK0 integrator only supports linear term");
  if (scheme != ETDRK0 && plan->term == TERM_NONE)
    return fail(TFSM_E_INVALID, "term not supported by engine: a nonlinear scheme needs a product term");
  if (n_points < 1) return fail(TFSM_E_INVALID, "n_integration_points must be >= 1");
  CoefArgs a;
  a.scheme = scheme;
  a.dt = dt;
  a.dt32 = (float)dt;
  a.hdt32 = (float)(0.5 * dt);
  a.M = n_points;
  a.radius = radius;
  a.modes = plan->modes;
  a.Bc = plan->Bc;
  a.L = plan->L;
  a.coef = plan->coef;
  a.cpk = plan->cpk;
  a.c5t = plan->c5t;
  a.ck01 = plan->ck01;
  a.c6t = plan->c6t;
  a.Lc = plan->Lc;
  a.coefc = plan->coefc;
  HIP_TRY(launch_coefs(a, (hipStream_t)stream), "coefficient launch");
  if (!plan->cplx) HIP_TRY(launch_pack_coefs(a, (hipStream_t)stream), "coefficient pack launch");
  plan->scheme = scheme;
  plan->dt = dt;
  plan->n_points = n_points;
  plan->radius = radius;
  return TFSM_OK;
}

int tfsm_plan_set_sample(tfsm_plan* p, int32_t b, const float* linear_coef, double length, void* stream) {
  if (!p) return fail(TFSM_E_INVALID, "null plan");
  if (b < 0 || b >= p->B) return fail(TFSM_E_INVALID, "sample index out of range");
  const int rows_per = p->per_len ? p->C : 1;
  if (p->Bc != p->B * rows_per) return fail(TFSM_E_INVALID, "the plan has shared coefficients (coef_batch 1)");
  if (length > 0 && !p->per_len) return fail(TFSM_E_INVALID, "per-sample lengths need a 1D plan created with them");
  hipStream_t st = (hipStream_t)stream;
  for (int r = b * rows_per; r < (b + 1) * rows_per; ++r) {
    if (length > 0) {
      const int n = p->n[0];
      const double d = length / n;
      HIP_TRY(launch_axis_row(p->kv[0] + (size_t)r * p->kv_bstride, n, (float)(1.0 / (n * d)), st), "axis row launch");
    }
    if (linear_coef || length > 0) {
      if (!linear_coef) return fail(TFSM_E_INVALID, "a new length needs the sample's linear coefficients");
      LinArgs la;
      la.D = p->D;
      for (int d = 0; d < 3; ++d) {
        la.n[d] = p->n[d];
        la.kv[d] = p->kv[d];
      }
      if (p->per_len) la.kv[0] = p->kv[0] + (size_t)r * p->kv_bstride;
      la.H = p->H;
      la.P = p->P;
      la.modes = p->modes;
      la.kv_bstride = 0;
      la.nterm = p->nlin;
      for (int t = 0; t < 4; ++t) {
        la.kind[t] = t < p->nlin ? p->lin_kind[t] : 0;
        la.dim[t] = p->lin_dim[t];
        la.order[t] = p->lin_order[t];
        la.cval[t] = t < p->nlin ? linear_coef[t] : 0.f;
      }
      la.coef = nullptr;
      la.Bc = 1;
      la.L = p->L + (size_t)r * p->modes;
      la.Lc = p->cplx ? p->Lc + (size_t)r * p->modes : nullptr;
      HIP_TRY(launch_linear_symbol(la, st), "linear symbol launch");
    }
    if (p->scheme >= 0) {
      CoefArgs a;
      a.scheme = p->scheme;
      a.dt = p->dt;
      a.dt32 = (float)p->dt;
      a.hdt32 = (float)(0.5 * p->dt);
      a.M = p->n_points;
      a.radius = p->radius;
      a.modes = p->modes;
      a.Bc = 1;
      a.L = p->L + (size_t)r * p->modes;
      a.coef = p->coef + (size_t)r * NCOEF * p->modes;
      a.cpk = p->cpk + (size_t)r * 2 * p->modes;
      a.c5t = p->c5t + (size_t)r * p->modes;
      a.ck01 = p->ck01 + (size_t)r * p->modes;
      a.c6t = p->c6t + (size_t)r * p->modes;
      a.Lc = p->cplx ? p->Lc + (size_t)r * p->modes : nullptr;
      a.coefc = p->cplx ? p->coefc + (size_t)r * NCOEF * p->modes : nullptr;
      HIP_TRY(launch_coefs(a, st), "coefficient launch");
      if (!p->cplx) HIP_TRY(launch_pack_coefs(a, st), "coefficient pack launch");
    }
  }
  return TFSM_OK;
}

int tfsm_plan_coefficients(tfsm_plan* p, int32_t slot, float* out, void* stream) {
  if (!p || !out) return fail(TFSM_E_INVALID, "null argument");
  if (slot < 0 || slot >= NCOEF) return fail(TFSM_E_INVALID, "coefficient slot out of range");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  const size_t bytes = p->modes * sizeof(float);
  for (int b = 0; b < p->Bc; ++b)
    HIP_TRY(hipMemcpyAsync(out + (size_t)b * p->modes, p->coef + ((size_t)b * NCOEF + slot) * p->modes, bytes,
                           hipMemcpyDeviceToDevice, (hipStream_t)stream),
            "coefficient copy");
  return TFSM_OK;
}

int tfsm_forward(tfsm_plan* p, const float* u, void* uh, int32_t nbatch, void* stream) {
  if (!p || !u || !uh) return fail(TFSM_E_INVALID, "null argument");
  if (int rc = check_nbatch(p, nbatch)) return rc;
  return xf_forward_blocks(p, u, (float2*)uh, (size_t)nbatch * p->C, (hipStream_t)stream);
}

int tfsm_inverse(tfsm_plan* p, const void* uh, float* u, int32_t nbatch, void* scratch, void* stream) {
  if (!p || !u || !uh) return fail(TFSM_E_INVALID, "null argument");
  if (int rc = check_nbatch(p, nbatch)) return rc;
  if (p->D > 1 && !scratch) return fail(TFSM_E_INVALID, "inverse transform needs scratch");
  const float scale = (float)(1.0 / (double)plan_npts(p));
  return xf_inverse_blocks(p, (const float2*)uh, (float2*)scratch, u, (size_t)nbatch * p->C, scale,
                           (hipStream_t)stream);
}

int32_t tfsm_plan_forward_fills(const tfsm_plan* p) { return p && fast_rows(p, p->D - 1) && p->P <= p->n[p->D - 1] ? 1 : 0; }

int tfsm_integrate_linear(tfsm_plan* p, const float* u, float* out, int32_t nsteps, void* scratch, void* stream) {
  if (!p || !u || !out || !scratch) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme != ETDRK0) return fail(TFSM_E_STATE, "the exact linear stepper (ETDRK0) is not the plan's scheme");
  if (nsteps < 0) return fail(TFSM_E_INVALID, "nsteps must be >= 0");
  if (int rc = check_nbatch(p, p->B)) return rc;
  hipStream_t st = (hipStream_t)stream;
  float2* W = (float2*)scratch;
  const int D = p->D, nl = p->n[D - 1];
  const size_t blk = (size_t)p->B * p->C;
  const float* E = p->coef + CS_E * p->modes;
  const float2* Ec = p->cplx ? p->coefc + CS_E * p->modes : nullptr;
  const float scale = (float)(1.0 / (double)plan_npts(p));
  if (D == 1 && fast_rows(p, 0) && !p->per_len) {
    HIP_TRY(launch_rows_linear(nl, u, out, (int)blk, scale, p->tw[0][0], E, Ec, p->coef_bstride(), p->C, nsteps, st),
            "linear row launch");
    return TFSM_OK;
  }
  if (D == 1 || !fast_cols(p, 0)) {  // the passes one by one
    int rc = xf_forward_blocks(p, u, W, blk, st);
    if (!rc) rc = step_impl(p, W, nsteps, nullptr, nullptr, 0, nullptr, st);
    return rc ? rc : xf_inverse_blocks(p, W, W, out, blk, scale, st);
  }
  const size_t rows = blk * p->modes / p->P, plane = D == 3 ? (size_t)p->n[1] * p->P : (size_t)p->P;
  HIP_TRY(xf_rows(p, GM_R2C, -1, u, (size_t)nl, W, (size_t)p->P, rows, 1.0f, st), "r2c launch");
  if (D == 3)
    HIP_TRY(xf_cols(p, 1, -1, W, W, blk * p->n[0], plane, (size_t)p->P, (size_t)p->H, st), "y fft launch");
  HIP_TRY(launch_cols_linear(p->n[0], W, blk, p->modes, plane, D == 3 ? (int)plane : p->H, p->tw[0][0], E, Ec,
                             p->coef_bstride(), p->C, nsteps, st),
          "linear column launch");
  if (D == 3)
    HIP_TRY(xf_cols(p, 1, +1, W, W, blk * p->n[0], plane, (size_t)p->P, (size_t)p->H, st), "y ifft launch");
  HIP_TRY(xf_rows(p, GM_C2R, +1, W, (size_t)p->P, out, (size_t)nl, rows, scale, st), "c2r launch");
  return TFSM_OK;
}

int tfsm_c2c(tfsm_plan* p, const void* in, void* out, int32_t nbatch, int32_t dir, void* stream) {
  if (!p || !in || !out) return fail(TFSM_E_INVALID, "null argument");
  if (dir != -1 && dir != 1) return fail(TFSM_E_INVALID, "dir must be -1 or +1");
  if (int rc = check_nbatch(p, nbatch)) return rc;
  hipStream_t st = (hipStream_t)stream;
  const size_t blocks = (size_t)nbatch * p->C;
  const int nl = p->n[p->D - 1];
  const float scale = dir > 0 ? (float)(1.0 / (double)plan_npts(p)) : 1.0f;
  size_t rows = blocks;
  for (int d = 0; d < p->D - 1; ++d) rows *= p->n[d];
  HIP_TRY(xf_rows(p, GM_C2C, dir, in, (size_t)nl, out, (size_t)nl, rows, scale, st), "row c2c launch");
  float2* o = (float2*)out;
  if (p->D == 2)
    HIP_TRY(xf_cols(p, 0, dir, o, o, blocks, (size_t)p->n[0] * nl, (size_t)nl, (size_t)nl, st), "column c2c launch");
  if (p->D == 3) {
    const size_t plane = (size_t)p->n[1] * nl;
    HIP_TRY(xf_cols(p, 1, dir, o, o, blocks * p->n[0], plane, (size_t)nl, (size_t)nl, st), "y c2c launch");
    HIP_TRY(xf_cols(p, 0, dir, o, o, blocks, (size_t)p->n[0] * plane, plane, plane, st), "x c2c launch");
  }
  return TFSM_OK;
}

int tfsm_half_to_full(tfsm_plan* p, const void* uh, void* full, int32_t nbatch, void* stream) {
  if (!p || !uh || !full) return fail(TFSM_E_INVALID, "null argument");
  if (int rc = check_nbatch(p, nbatch)) return rc;
  ConvArgs a;
  a.D = p->D;
  for (int d = 0; d < 3; ++d) a.n[d] = p->n[d];
  a.H = p->H;
  a.P = p->P;
  a.nblk = (size_t)nbatch * p->C;
  HIP_TRY(launch_half_to_full((const float2*)uh, (float2*)full, a, (hipStream_t)stream), "half_to_full launch");
  return TFSM_OK;
}

int tfsm_full_to_half(tfsm_plan* p, const void* full, void* uh, int32_t nbatch, void* stream) {
  if (!p || !uh || !full) return fail(TFSM_E_INVALID, "null argument");
  if (int rc = check_nbatch(p, nbatch)) return rc;
  ConvArgs a;
  a.D = p->D;
  for (int d = 0; d < 3; ++d) a.n[d] = p->n[d];
  a.H = p->H;
  a.P = p->P;
  a.nblk = (size_t)nbatch * p->C;
  HIP_TRY(launch_full_to_half((const float2*)full, (float2*)uh, a, (hipStream_t)stream), "full_to_half launch");
  return TFSM_OK;
}

int tfsm_plan_add_source(tfsm_plan* p, const float* src, int32_t src_batch, int32_t src_channels, float coef,
                         void* stream) {
  if (!p || !src) return fail(TFSM_E_INVALID, "null argument");
  if (!(src_batch == 1 || src_batch == p->B) || !(src_channels == 1 || src_channels == p->C))
    return fail(TFSM_E_INVALID, "source batch/channels must be 1 or match the state");
  if (p->src && (src_batch != p->srcB || src_channels != p->srcC))
    return fail(TFSM_E_INVALID, "all explicit sources of one operator must have the same shape");
  hipStream_t st = (hipStream_t)stream;
  const size_t total = (size_t)src_batch * src_channels * p->modes;
  float2* spec = nullptr;
  HIP_TRY(hipMalloc(&spec, total * sizeof(float2)), "source spectrum scratch");
  // forward transform of the source with a plan-compatible batch of src_batch blocks of src_channels
  const int saveC = p->C;
  p->C = src_channels;
  int rc = tfsm_forward(p, src, spec, src_batch, stream);
  p->C = saveC;
  const bool first = p->src == nullptr;
  if (!rc && first) rc = dev_alloc(p, &p->src, total, "source spectrum");
  if (!rc) {
    hipError_t e = launch_accum_source(p->src, spec, coef, total, first ? 1 : 0, st);
    if (e != hipSuccess) rc = hip_fail(e, "source accumulate launch");
  }
  (void)hipStreamSynchronize(st);
  (void)hipFree(spec);
  if (rc) return rc;
  p->srcB = src_batch;
  p->srcC = src_channels;
  if (p->D == 2) {
    // columns (last-axis frequencies) where the accumulated source has a nonzero mode: the fused
    // column kernels skip the source loads elsewhere (adding an exact zero changes nothing)
    std::vector<float2> h(total);
    HIP_TRY(hipMemcpy(h.data(), p->src, total * sizeof(float2), hipMemcpyDeviceToHost), "source spectrum download");
    std::vector<unsigned char> cols(p->P, 0);
    for (size_t e = 0; e < total; ++e)
      if (h[e].x != 0.f || h[e].y != 0.f) cols[e % p->P] = 1;
    if (!p->src_cols) rc = dev_alloc(p, &p->src_cols, (size_t)p->P, "source column flags");
    if (rc) return rc;
    HIP_TRY(hipMemcpy(p->src_cols, cols.data(), cols.size(), hipMemcpyHostToDevice), "source column flags upload");
    p->src_bits_ok = p->P <= 32 * Col2Args::SRC_BIT_WORDS;
    for (int w = 0; w < Col2Args::SRC_BIT_WORDS; ++w) p->src_bits[w] = 0;
    if (p->src_bits_ok)
      for (int k = 0; k < p->P; ++k)
        if (cols[k]) p->src_bits[k >> 5] |= 1u << (k & 31);
  }
  return TFSM_OK;
}

int tfsm_plan_add_force(tfsm_plan* p, const float* force, int32_t force_batch, int32_t force_channels, float coef,
                        void* stream) {
  if (!p || !force) return fail(TFSM_E_INVALID, "null argument");
  if (p->term != TERM_NSP)
    return fail(TFSM_E_INVALID, "an external force belongs to NSPressureConvection (velocity-form Navier-Stokes)");
  if (!(force_batch == 1 || force_batch == p->B) || !(force_channels == 1 || force_channels == p->C))
    return fail(TFSM_E_INVALID, "force batch/channels must be 1 or match the state");
  if (p->force && (force_batch != p->forceB || force_channels != p->forceC))
    return fail(TFSM_E_INVALID, "all explicit sources of one force must have the same shape");
  hipStream_t st = (hipStream_t)stream;
  const size_t total = (size_t)force_batch * force_channels * p->modes;
  float2* spec = nullptr;
  HIP_TRY(hipMalloc(&spec, total * sizeof(float2)), "force spectrum scratch");
  const int saveC = p->C;
  p->C = force_channels;
  int rc = tfsm_forward(p, force, spec, force_batch, stream);
  p->C = saveC;
  const bool first = p->force == nullptr;
  if (!rc && first) rc = dev_alloc(p, &p->force, total, "force spectrum");
  if (!rc) {
    hipError_t e = launch_accum_source(p->force, spec, coef, total, first ? 1 : 0, st);
    if (e != hipSuccess) rc = hip_fail(e, "force accumulate launch");
  }
  (void)hipStreamSynchronize(st);
  (void)hipFree(spec);
  if (rc) return rc;
  p->forceB = force_batch;
  p->forceC = force_channels;
  // the forced core masks the integrator's stage tensors in place: only the unfused path does that
  p->fused_ok = false;
  p->persistent = false;
  if (!p->general || p->genf) {
    p->general = true;
    p->genf = p->genf_ok = p->gf_row = p->gf_col = false;
    gen_layout(p);
  }
  return TFSM_OK;
}

int tfsm_step(tfsm_plan* p, void* uh, int32_t nsteps, const int32_t* rec_slot, void* traj, int32_t T, void* ws,
              void* stream) {
  if (!p || !uh) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (nsteps < 0) return fail(TFSM_E_INVALID, "nsteps must be >= 0");
  if (rec_slot && (!traj || T < 1)) return fail(TFSM_E_INVALID, "recording needs a trajectory buffer");
  return step_impl(p, uh, nsteps, rec_slot, traj, T, ws, (hipStream_t)stream);
}

int tfsm_step_noalloc(tfsm_plan* p, void* uh, int32_t nsteps, const int32_t* rec_slot, void* traj, int32_t T,
                      void* stream) {
  if (!p || !uh) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (nsteps < 0) return fail(TFSM_E_INVALID, "nsteps must be >= 0");
  if (rec_slot && (!traj || T < 1)) return fail(TFSM_E_INVALID, "recording needs a trajectory buffer");
  if (p->ws_bytes > (size_t)TFSM_NOALLOC_SCRATCH_BYTES)
    return fail(TFSM_E_INVALID, "the plan's workspace (" + std::to_string(p->ws_bytes) +
                                    " bytes) exceeds the static scratch of tfsm_step_noalloc (" +
                                    std::to_string((long long)TFSM_NOALLOC_SCRATCH_BYTES) +
                                    " bytes): use tfsm_step with a caller workspace or a smaller batch");
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev), "current device");
  if (dev != p->device) return fail(TFSM_E_INVALID, "the plan's device must be the current device");
  void* ws = nullptr;
  const int rc = scratch_on_device(dev, &ws);
  if (rc) return rc;
  return step_impl(p, uh, nsteps, rec_slot, traj, T, ws, (hipStream_t)stream);
}

int tfsm_step_varying(tfsm_plan* p, void* uh, const int32_t* nsteps_per_sample, int32_t max_steps, void* ws,
                      void* stream) {
  if (!p || !uh || !nsteps_per_sample || !ws) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (max_steps < 0) return fail(TFSM_E_INVALID, "max_steps must be >= 0");
  if (p->scheme == ETDRK0) return fail(TFSM_E_INVALID, "per-sample step counts need a nonlinear plan");
  if (p->term == TERM_KS && (p->D == 1 || p->ks_mean))
    return fail(TFSM_E_INVALID, "per-sample step counts are not available for KSConvection in 1D or with remove_mean "
                                "(its mean couples the samples)");
  if (p->D == 1) {
    Run1Args a = run1_args(p, (float2*)uh, (char*)ws);
    a.nsteps = max_steps;
    a.nsteps_per = nsteps_per_sample;
    HIP_TRY(launch_run1d(a, (hipStream_t)stream), "1D stepper launch");
    return TFSM_OK;
  }
  return step_impl(p, uh, max_steps, nullptr, nullptr, 0, ws, (hipStream_t)stream, nsteps_per_sample);
}

int tfsm_apply(tfsm_plan* p, const void* uh, void* out, void* ws, void* stream) {
  if (!p || !uh || !out) return fail(TFSM_E_INVALID, "null argument");
  hipStream_t st = (hipStream_t)stream;
  const bool have_nl = p->term != TERM_NONE;
  const bool have_lin = p->nlin > 0;
  float2* U = (float2*)uh;
  if (have_nl) {
    if (!ws) return fail(TFSM_E_INVALID, "workspace pointer is null");
    if (p->general || p->l1) {
      if (int rc = eval_nonlinear(p, U, (char*)ws, st)) return rc;
    } else if (p->D == 1 && p->term == TERM_KS) {
      Run1Args a = run1_args(p, U, (char*)ws);
      float2* Nr = (float2*)((char*)ws + p->off_N);
      float2* dc = p->ks_mean ? (float2*)((char*)ws + p->off_DC) : nullptr;
      HIP_TRY(launch_k1_eval_ks(a, U, Nr, st), "1D product launch");
      if (dc) HIP_TRY(launch_ks_dc(Nr, a.B, (size_t)p->P, 1, 0, dc, st), "batch-mean launch");
      HIP_TRY(launch_k1_stage(a, ST_EVAL, Nr, dc, (float2*)((char*)ws + p->off_S), st), "1D stage launch");
    } else if (p->D == 1) {
      Run1Args a = run1_args(p, U, (char*)ws);
      a.eval_only = 1;
      a.nsteps = 1;
      HIP_TRY(launch_run1d(a, st), "1D evaluation launch");
    } else {
      int rc = run_eval(p, U, (char*)ws, ST_PRO, 0, p->B, st);
      if (!rc) rc = run_eval(p, U, (char*)ws, ST_EVAL, 0, p->B, st);
      if (rc) return rc;
    }
  }
  const float2* Nv = have_nl ? (const float2*)((char*)ws + p->off_A1) : nullptr;
  if (p->cplx)
    HIP_TRY(launch_apply_linear_c(U, Nv, p->Lc, p->Bc > 1 ? p->modes : 0, p->modes, p->C, p->state_elems(), have_lin,
                                  have_nl, (float2*)out, st),
            "apply launch");
  else
    HIP_TRY(launch_apply_linear(U, Nv, p->L, p->Bc > 1 ? p->modes : 0, p->modes, p->C, p->state_elems(), have_lin,
                                have_nl, (float2*)out, st),
            "apply launch");
  return TFSM_OK;
}

int tfsm_spectral_map(tfsm_plan* p, int32_t op, float coef, const void* in, void* out, void* stream) {
  if (!p || !in || !out) return fail(TFSM_E_INVALID, "null argument");
  MapArgs a;
  a.op = op;
  a.D = p->D;
  a.B = p->B;
  switch (op) {
    case MAP_DEALIAS: a.cin = p->C; a.cout = p->C; break;
    case MAP_DIV: a.cin = p->D; a.cout = 1; break;
    case MAP_GRAD: a.cin = 1; a.cout = p->D; break;
    case MAP_CURL:
      if (p->D < 2) return fail(TFSM_E_INVALID, "curl operator only works for 2D or 3D vector field");
      a.cin = p->D; a.cout = p->D == 2 ? 1 : 3;
      break;
    case MAP_V2V:
      if (p->D != 2) return fail(TFSM_E_INVALID, "Only vorticity in 2Dmesh is supported");
      a.cin = 1; a.cout = 2;
      break;
    case MAP_PRESSURE: a.cin = p->D; a.cout = 1; break;
    case MAP_CONSDIV: a.cin = p->D * p->D; a.cout = p->D; break;
    default: return fail(TFSM_E_INVALID, "unknown spectral map");
  }
  for (int d = 0; d < 3; ++d) {
    a.n[d] = p->n[d];
    a.kv[d] = p->kv[d];
    a.kmax[d] = p->kmax[d];
  }
  if (p->kv_bstride) return fail(TFSM_E_INVALID, "spectral maps need shared lengths");
  a.H = p->H;
  a.P = p->P;
  a.modes = p->modes;
  a.coef = coef;
  a.in = (const float2*)in;
  a.out = (float2*)out;
  HIP_TRY(launch_spectral_map(a, (hipStream_t)stream), "spectral map launch");
  return TFSM_OK;
}

int tfsm_pointwise_products(tfsm_plan* p, const float* u, float* out, void* stream) {
  if (!p || !u || !out) return fail(TFSM_E_INVALID, "null argument");
  size_t npts = 1;
  for (int d = 0; d < p->D; ++d) npts *= p->n[d];
  HIP_TRY(launch_pointwise_products(u, out, p->B, p->C, npts, (hipStream_t)stream), "products launch");
  return TFSM_OK;
}

int tfsm_rk_combine(tfsm_plan* p, void* out, const void* x, const void* const* ks, const float* coefs, int32_t nk,
                    float dt, void* stream) {
  if (!p || !out || !x || (nk > 0 && (!ks || !coefs))) return fail(TFSM_E_INVALID, "null argument");
  if (nk < 0 || nk > RK_MAX_TERMS) return fail(TFSM_E_INVALID, "at most 8 stage terms");
  RkArgs a;
  a.x = (const float2*)x;
  for (int i = 0; i < RK_MAX_TERMS; ++i) {
    a.k[i] = i < nk ? (const float2*)ks[i] : nullptr;
    a.c[i] = i < nk ? coefs[i] : 0.f;
    if (i < nk && !ks[i]) return fail(TFSM_E_INVALID, "null stage pointer");
  }
  a.nk = nk;
  a.dt = dt;
  a.out = (float2*)out;
  a.total = p->state_elems();
  HIP_TRY(launch_rk_combine(a, (hipStream_t)stream), "rk combine launch");
  return TFSM_OK;
}

int tfsm_solve(tfsm_plan* p, const void* uh, void* out, void* stream) {
  if (!p || !uh || !out) return fail(TFSM_E_INVALID, "null argument");
  if (p->nlin == 0) return fail(TFSM_E_INVALID, "solve needs a linear operator");
  if (p->cplx)
    HIP_TRY(launch_apply_linear_c((const float2*)uh, nullptr, p->Lc, p->Bc > 1 ? p->modes : 0, p->modes, p->C,
                                  p->state_elems(), 2, 0, (float2*)out, (hipStream_t)stream),
            "solve launch");
  else
    HIP_TRY(launch_apply_linear((const float2*)uh, nullptr, p->L, p->Bc > 1 ? p->modes : 0, p->modes, p->C,
                                p->state_elems(), 2, 0, (float2*)out, (hipStream_t)stream),
            "solve launch");
  return TFSM_OK;
}

int tfsm_launch_pass(tfsm_plan* p, void* uh, void* ws, int32_t pass_id, int32_t stage, int32_t sub, void* stream) {
  if (!p || !uh || !ws) return fail(TFSM_E_INVALID, "null argument");
  if (p->general) return fail(TFSM_E_INVALID, "the plan has no fixed-size fused passes");
  hipStream_t st = (hipStream_t)stream;
  // the launches cover sub-batch `sub`, exactly as tfsm_step launches them
  const int sb = (p->sub_batch > 0 && p->sub_batch < p->B) ? p->sub_batch : p->B;
  if (sub < 0 || (int64_t)sub * sb >= p->B) return fail(TFSM_E_INVALID, "sub-batch index out of range");
  const int b0 = sub * sb;
  const int nb = (p->B - b0) < sb ? (p->B - b0) : sb;
  if (p->D == 2) {
    if (p->term == TERM_NONE) return fail(TFSM_E_INVALID, "no product term");
    if (pass_id == 0) return launch_row(p, (char*)ws, b0, nb, st);
    if (pass_id == 1) {
      if (stage < ST_PRO || stage > ST_EVAL) return fail(TFSM_E_INVALID, "bad stage");
      if (stage != ST_PRO && p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
      return launch_col(p, (float2*)uh, (char*)ws, stage, b0, nb, st);
    }
  }
  if (p->D == 3) {
    if (p->term == TERM_NONE) return fail(TFSM_E_INVALID, "no product term");
    if (stage < ST_PRO || stage > ST_EVAL) return fail(TFSM_E_INVALID, "bad stage");
    if (stage != ST_PRO && p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
    // one whole evaluation (4 kernels) per call; pass ids 0/1 are not split for 3D
    if (pass_id == 3) return run3d_eval(p, (float2*)uh, (char*)ws, stage, b0, nb, st);
    if (pass_id >= 4 && pass_id <= 7)
      return run3d_eval(p, (float2*)uh, (char*)ws, stage, b0, nb, st, 1 << (pass_id - 4));
  }
  if (p->D == 1 && pass_id == 2) {
    if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
    if (p->term == TERM_KS) return fail(TFSM_E_INVALID, "1D KSConvection steps stage by stage (tfsm_step)");
    if (p->l1) return fail(TFSM_E_INVALID, "long 1D meshes step stage by stage (tfsm_step)");
    Run1Args a = run1_args(p, (float2*)uh, (char*)ws);
    a.nsteps = 1;
    HIP_TRY(launch_run1d(a, st), "1D stepper launch");
    return TFSM_OK;
  }
  return fail(TFSM_E_INVALID, "unknown pass for this plan");
}

int tfsm_launch_pass_timed(tfsm_plan* p, void* uh, void* ws, int32_t pass_id, int32_t stage, int32_t sub,
                           void* ev_start, void* ev_stop, void* stream) {
  if (!ev_start || !ev_stop) return fail(TFSM_E_INVALID, "null event");
  g_launch_ev[0] = (hipEvent_t)ev_start;
  g_launch_ev[1] = (hipEvent_t)ev_stop;
  const int rc = tfsm_launch_pass(p, uh, ws, pass_id, stage, sub, stream);
  g_launch_ev[0] = g_launch_ev[1] = nullptr;
  return rc;
}

int64_t tfsm_plan_adjoint_workspace_bytes(const tfsm_plan* plan) {
  return plan ? (int64_t)adj_layout(plan).total : 0;
}

int tfsm_adjoint_prepare(tfsm_plan* p, int32_t grad_term, void* stream) {
  if (!p) return fail(TFSM_E_INVALID, "null plan");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (p->scheme != ETDRK1 && p->scheme != ETDRK2 && p->scheme != SETDRK1 && p->scheme != SETDRK2 &&
      p->scheme != SETDRK4)
    return fail(TFSM_E_INVALID, "term not supported by engine: the adjoint covers ETDRK1/2 and SETDRK1/2/4");
  if (!(p->term == TERM_CONV || (p->term == TERM_VC && p->D == 2)))
    return fail(TFSM_E_INVALID,
                "term not supported by engine: the adjoint covers Convection (1D, 2D, 3D) and VorticityConvection");
  // explicit sources are constant: they enter the recomputed states but no Jacobian
  if (p->cplx) return fail(TFSM_E_INVALID, "term not supported by engine: the adjoint needs a real linear symbol");
  if (p->force) return fail(TFSM_E_INVALID, "term not supported by engine: the adjoint of a forced NSPressureConvection");
  if (p->per_len) return fail(TFSM_E_INVALID, "term not supported by engine: the adjoint needs shared lengths");
  if (grad_term < -1 || grad_term >= p->nlin) return fail(TFSM_E_INVALID, "grad_term out of range");
  hipStream_t st = (hipStream_t)stream;
  int rc = TFSM_OK;
  if (!p->dcoef) rc = dev_alloc(p, &p->dcoef, (size_t)p->Bc * ADJ_NDCOEF * p->modes, "adjoint coefficient table");
  if (!rc && !p->sym) rc = dev_alloc(p, &p->sym, p->modes, "adjoint symbol");
  if (rc) return rc;
  if (p->scheme == SETDRK4)
    HIP_TRY(launch_adj_dcoefs4(p->L, p->modes, p->Bc, p->dt, p->n_points, p->radius, p->dcoef, st),
            "adjoint coefficient launch");
  else
    HIP_TRY(launch_adj_dcoefs(p->L, p->modes, p->Bc, p->dt, p->dcoef, st), "adjoint coefficient launch");
  if (grad_term >= 0) HIP_TRY(launch_adj_sym(adj_args(p), p->lin_kind[grad_term], p->sym, st), "adjoint symbol launch");
  p->adj_term = grad_term;
  p->adj_scheme = p->scheme;
  return TFSM_OK;
}

int tfsm_adjoint_step(tfsm_plan* p, void* u, const void* ubar_next, void* ubar, double* grad, void* ws, void* wsa,
                      void* stream) {
  if (!p || !u || !ubar_next || !ubar || !ws || !wsa) return fail(TFSM_E_INVALID, "null argument");
  if (p->adj_term < -1 || p->adj_scheme != p->scheme) return fail(TFSM_E_STATE, "tfsm_adjoint_prepare not called");
  if (ubar == ubar_next || ubar == u) return fail(TFSM_E_INVALID, "ubar must not alias the inputs");
  hipStream_t st = (hipStream_t)stream;
  char* W = (char*)ws;
  char* A = (char*)wsa;
  const AdjLayout l = adj_layout(p);
  float2* U = (float2*)u;
  const float2* Ubn = (const float2*)ubar_next;
  float2* Ubo = (float2*)ubar;
  float2* A1 = (float2*)(W + p->off_A1);
  float2* Aa = (float2*)(A + l.Aa);
  float2* N0s = (float2*)(A + l.N0s);
  float2* T1 = (float2*)(A + l.T1);
  float2* Jv = (float2*)(A + l.Jv);
  float2* Ab = (float2*)(A + l.Ab);
  float2* Nb = (float2*)(A + l.Nb);
  const bool want = grad && p->adj_term >= 0;
  const size_t sbytes = p->state_elems() * sizeof(float2);
  if (adj_fused(p)) return adj_step_fused(p, U, Ubn, Ubo, grad, W, A, st);
  if (p->scheme == SETDRK4) return adjoint_step4(p, U, Ubn, Ubo, grad, W, A, st);
  AdjGradArgs g = grad_args(p, A, grad);
  int rc = eval_nonlinear(p, U, W, st);
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(N0s, A1, sbytes, hipMemcpyDeviceToDevice, st), "adjoint copy");
  AdjStageArgs s = stage_args(p, ADJ_PRE);
  if (s.two_stage) {
    s.op = ADJ_STAGE_A;
    s.X0 = U;
    s.X1 = N0s;
    s.Y0 = Aa;
    HIP_TRY(launch_adj_stage(s, st), "adjoint stage launch");
    rc = eval_nonlinear(p, Aa, W, st);  // Na -> A1
    if (rc) return rc;
    s = stage_args(p, ADJ_PRE);
    s.X0 = Ubn;
    s.Y0 = T1;
    HIP_TRY(launch_adj_stage(s, st), "adjoint stage launch");
    rc = adj_jt(p, Aa, T1, Jv, A, st);
    if (rc) return rc;
    s = stage_args(p, ADJ_MID);
    s.X0 = Ubn;
    s.X1 = Jv;
    s.Y0 = Ab;
    s.Y1 = Nb;
    HIP_TRY(launch_adj_stage(s, st), "adjoint stage launch");
    rc = adj_jt(p, U, Nb, Jv, A, st);
    if (rc) return rc;
    s = stage_args(p, ADJ_POST);
    s.X0 = Ab;
    grad_term(g, Ubn, A1, D_C2, 1.f);
    grad_term(g, Ubn, N0s, D_C2, -1.f);
  } else {
    s.X0 = Ubn;
    s.Y0 = T1;
    HIP_TRY(launch_adj_stage(s, st), "adjoint stage launch");
    rc = adj_jt(p, U, T1, Jv, A, st);
    if (rc) return rc;
    s = stage_args(p, ADJ_POST);
    s.X0 = Ubn;
  }
  s.X1 = Jv;
  s.Y0 = Ubo;
  HIP_TRY(launch_adj_stage(s, st), "adjoint stage launch");
  grad_term(g, s.X0, U, D_E, 1.f);
  grad_term(g, s.X0, N0s, D_C1, 1.f);
  if (want) HIP_TRY(launch_adj_grad(g, st), "adjoint gradient launch");
  return TFSM_OK;
}

}  // extern "C"

namespace {
// nsteps of step_impl (optionally with per-sample counts) captured into an instantiated graph
int graph_capture(tfsm_plan* p, void* uh, int nsteps, const int* act, void* ws, void* stream, tfsm_graph** out) {
  *out = nullptr;
  hipStream_t cap = nullptr;
  HIP_TRY(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking), "capture stream");
  // order the capture stream after the caller's stream so that setup work is visible
  hipEvent_t ev = nullptr;
  HIP_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "capture event");
  HIP_TRY(hipEventRecord(ev, (hipStream_t)stream), "capture event record");
  HIP_TRY(hipStreamWaitEvent(cap, ev, 0), "capture wait");
  HIP_TRY(hipStreamSynchronize(cap), "capture sync");
  (void)hipEventDestroy(ev);
  tfsm_graph* g = new tfsm_graph();
  hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) {
    delete g;
    (void)hipStreamDestroy(cap);
    return hip_fail(e, "begin capture");
  }
  int rc = step_impl(p, uh, nsteps, nullptr, nullptr, 0, ws, cap, act);
  e = hipStreamEndCapture(cap, &g->graph);
  if (rc == TFSM_OK && e != hipSuccess) rc = hip_fail(e, "end capture");
  if (rc == TFSM_OK) {
    e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) rc = hip_fail(e, "graph instantiate");
  }
  (void)hipStreamDestroy(cap);
  if (rc) {
    tfsm_graph_destroy(g);
    return rc;
  }
  *out = g;
  return TFSM_OK;
}
}  // namespace

extern "C" {

int tfsm_graph_create(tfsm_plan* p, void* uh, int32_t nsteps, void* ws, void* stream, tfsm_graph** out) {
  if (!p || !uh || !out) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (nsteps < 1) return fail(TFSM_E_INVALID, "a graph needs nsteps >= 1");
  return graph_capture(p, uh, nsteps, nullptr, ws, stream, out);
}

int tfsm_graph_create_varying(tfsm_plan* p, void* uh, const int32_t* nsteps_per_sample, int32_t max_steps, void* ws,
                              void* stream, tfsm_graph** out) {
  if (!p || !uh || !nsteps_per_sample || !ws || !out) return fail(TFSM_E_INVALID, "null argument");
  if (p->scheme < 0) return fail(TFSM_E_STATE, "no scheme set on the plan");
  if (max_steps < 1) return fail(TFSM_E_INVALID, "a graph needs max_steps >= 1");
  if (p->D < 2 || p->scheme == ETDRK0) return fail(TFSM_E_INVALID, "per-sample step graphs need a nonlinear 2D or 3D plan");
  if (p->term == TERM_KS && p->ks_mean)
    return fail(TFSM_E_INVALID, "per-sample step counts are not available for KSConvection with remove_mean "
                                "(its mean couples the samples)");
  return graph_capture(p, uh, max_steps, nsteps_per_sample, ws, stream, out);
}

int tfsm_graph_launch(tfsm_graph* g, void* stream) {
  if (!g || !g->exec) return fail(TFSM_E_INVALID, "null graph");
  HIP_TRY(hipGraphLaunch(g->exec, (hipStream_t)stream), "graph launch");
  return TFSM_OK;
}

int tfsm_graph_destroy(tfsm_graph* g) {
  if (!g) return TFSM_OK;
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  delete g;
  return TFSM_OK;
}

}  // extern "C"
