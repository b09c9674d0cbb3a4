// Bounded unit kernels for the reactor's device components (right-hand side,
// analytic Jacobian, LU factor/solve, BDF coefficients, Nordsieck order changes).
// The same file compiles for the GPU with hipcc and for the CPU with the serial
// stand-in under tests/cpu_emulation, so tests can compare the two bit for bit.
// Every kernel runs a fixed amount of work per lane.
#include <vector>

#include "../../pelelm_amd/csrc/reactor_bdf.hip"

#ifndef UNIT_HOST
#define UNIT_DEV_ALLOC(p, n) (void)hipMalloc((void**)&(p), (n))
#define UNIT_DEV_FREE(p) (void)hipFree(p)
#define UNIT_H2D(d, h, n) (void)hipMemcpy((d), (h), (n), hipMemcpyHostToDevice)
#define UNIT_D2H(h, d, n) (void)hipMemcpy((h), (d), (n), hipMemcpyDeviceToHost)
#define UNIT_SYNC() (void)hipDeviceSynchronize()
#else
#include <cstdlib>
thread_local Idx3 threadIdx, blockIdx, blockDim, gridDim;
#define UNIT_DEV_ALLOC(p, n) (p) = (decltype(p))std::malloc(n)
#define UNIT_DEV_FREE(p) std::free(p)
#define UNIT_H2D(d, h, n) std::memcpy((d), (h), (n))
#define UNIT_D2H(h, d, n) std::memcpy((h), (d), (n))
#define UNIT_SYNC()
#endif

namespace pelelm {
namespace {

// in:  y [ncell][N1], t, rE0, fH per cell; out: f [ncell][N1], Tsol
template <class M>
__global__ void k_rhs(const double* y, const double* t, const double* rE0, const double* fH, const double* fy,
                      double* f, double* Tsol, double* ws, long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  WS w{ws + (c >> 6) * (long)S::TOTAL * 64 + (c & 63)};
  for (int k = 0; k < N1 - 1; ++k) w[S::FY + k] = fy[c * (N1 - 1) + k];
  double yy[N1], ff[N1], T;
  for (int i = 0; i < N1; ++i) yy[i] = y[c * N1 + i];
  rhs<M>(yy, t[c], w, rE0[c], fH[c], ff, T);
  for (int i = 0; i < N1; ++i) f[c * N1 + i] = ff[i];
  Tsol[c] = T;
}

// Lanes with (lane % 3 != 0) evaluate the Jacobian at (y, T, fT), factor I - gamma J and
// solve for b; every lane carries a live vector through the branch and writes it back.
template <class M>
__global__ void k_jac_lu(const double* y, const double* T, const double* fT, const double* gamma,
                         const double* b, double* J, double* x, double* keep_out, int* sing, double* ws, double* mats,
                         long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  WS w{ws + (c >> 6) * (long)S::TOTAL * 64 + (c & 63)};
  const CM mat = cell_mat<M>(mats, c);
  double keep[N1];
  for (int i = 0; i < N1; ++i) keep[i] = y[c * N1 + i] * 3.0 + (double)c;
  // a private array indexed with a run-time value (so it lives in scratch) and a full
  // lane state, both live across the outlined calls below
  double dyn[8];
  const int idx = (int)(c * 7 % 8);
  for (int i = 0; i < 8; ++i) dyn[i] = (double)(c * 8 + i);
  dyn[idx] += 0.5;
  Lane<M> st;
  st.ws.p = ws;
  for (int i = 0; i < 6; ++i) st.tq[i] = (double)(c + i);
  for (int i = 0; i < LMAX; ++i) st.l[i] = (double)(2 * c + i);
  for (int i = 0; i <= LMAX; ++i) st.tau[i] = (double)(3 * c + i);
  st.q = 1 + (int)(c % 4);
  int sg = -1;
  if ((threadIdx.x % 3) != 0) {
    double yy[N1];
    for (int i = 0; i < N1; ++i) yy[i] = y[c * N1 + i];
    for (int k = 0; k < N1 - 1; ++k) w[S::FY + k] = 0.0;   // no species forcing
    jacobian<M>(yy, T[c], fT[c], w);
    for (int e = 0; e < N1 * N1; ++e) mat[MatSlots<N1>::JS + e] = w[S::JS + e];
    sg = lu_factor<N1, double>(mat, gamma[c]);
    for (int i = 0; i < N1; ++i) mat[MatSlots<N1>::B + i] = b[c * N1 + i];
    lu_solve<N1>(mat, MatSlots<N1>::B, MatSlots<N1>::X);
    for (int i = 0; i < N1; ++i) x[c * N1 + i] = mat[MatSlots<N1>::X + i];
    for (int e = 0; e < N1 * N1; ++e) J[c * N1 * N1 + e] = w[S::JS + e];
  }
  sing[c] = sg;
  for (int i = 0; i < N1; ++i) keep_out[c * N1 + i] = keep[i];
  // private state after the calls: dyn[0..7], tq[q], l[q], tau[q+1]
  double chk = 0.0;
  for (int i = 0; i < 8; ++i) chk += dyn[(idx + i) & 7] * (double)(i + 1);
  keep_out[ncell * N1 + c * 4 + 0] = chk;
  keep_out[ncell * N1 + c * 4 + 1] = st.tq[st.q];
  keep_out[ncell * N1 + c * 4 + 2] = st.l[st.q];
  keep_out[ncell * N1 + c * 4 + 3] = st.tau[st.q + 1];
}

// BDF coefficient / Nordsieck logic of one lane: set_coeffs for given (q, h, tau,
// qwait, nst, gammap), then an order increase and decrease on a given history.
// scal in : [q, qwait, nst, qmax, h, hscale, gammap, tau1..tau6]   (13 doubles)
// out     : l[0..5], tq[1..5], gamma, gamrat, rl1, zn after increase (6*N1), after decrease
template <class M>
__global__ void k_coeffs(const double* scal, const double* zn_in, double* out, double* ws, long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  Lane<M> st;
  st.ws.p = ws + (c >> 6) * (long)S::TOTAL * 64 + (c & 63);
  const double* s = scal + c * 13;
  st.q = (int)s[0];
  st.qwait = (int)s[1];
  st.nst = (long)s[2];
  st.qmax = (int)s[3];
  st.h = s[4];
  st.hscale = s[5];
  st.gammap = s[6];
  st.tau[0] = 0.0;
  for (int i = 1; i <= LMAX; ++i) st.tau[i] = s[6 + i];
  for (int i = 0; i < 6; ++i) st.tq[i] = -1.0;       // tq[1], tq[3] are only set when qwait == 1
  for (int i = 0; i < LMAX; ++i) st.l[i] = -1.0;
  st.L = st.q + 1;
  st.set_coeffs();
  double* o = out + c * (6 + 5 + 3 + 12 * N1);
  for (int i = 0; i < 6; ++i) o[i] = (i <= st.q) ? st.l[i] : 0.0;
  for (int i = 1; i <= 5; ++i) o[5 + i] = st.tq[i];
  o[11] = st.gamma;
  o[12] = st.gamrat;
  o[13] = st.rl1;
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) st.zn(j, i) = zn_in[(c * LMAX + j) * N1 + i];
  if (st.q < st.qmax) {
    st.L = st.q + 1;
    st.increase_bdf();
  }
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) o[14 + j * N1 + i] = st.zn(j, i);
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) st.zn(j, i) = zn_in[(c * LMAX + j) * N1 + i];
  if (st.q > 1) st.decrease_bdf();
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) o[14 + (LMAX + j) * N1 + i] = st.zn(j, i);
}

template <class T>
T* dev_copy(const T* h, size_t n) {
  T* d = nullptr;
  UNIT_DEV_ALLOC(d, n * sizeof(T));
  UNIT_H2D(d, h, n * sizeof(T));
  return d;
}
template <class T>
T* dev_zero(size_t n) {
  T* d = nullptr;
  UNIT_DEV_ALLOC(d, n * sizeof(T));
  std::vector<T> z(n, T(0));
  UNIT_H2D(d, z.data(), n * sizeof(T));
  return d;
}

template <class M>
int unit_rhs_t(long n, const double* y, const double* t, const double* rE0, const double* fH, const double* fy,
               double* f, double* T) {
  constexpr int N1 = M::N1;
  const long nw = (n + 63) / 64;
  double *dy = dev_copy(y, n * N1), *dt = dev_copy(t, n), *de = dev_copy(rE0, n), *dh = dev_copy(fH, n);
  double *dfy = dev_copy(fy, n * (N1 - 1)), *df = dev_zero<double>(n * N1), *dT = dev_zero<double>(n);
  double* ws = dev_zero<double>(nw * Slots<N1>::TOTAL * 64);
  hipLaunchKernelGGL(k_rhs<M>, dim3((unsigned)nw), dim3(64), 0, nullptr, dy, dt, de, dh, dfy, df, dT, ws, n);
  UNIT_SYNC();
  UNIT_D2H(f, df, n * N1 * sizeof(double));
  UNIT_D2H(T, dT, n * sizeof(double));
  for (void* p : {(void*)dy, (void*)dt, (void*)de, (void*)dh, (void*)dfy, (void*)df, (void*)dT, (void*)ws})
    UNIT_DEV_FREE(p);
  return 0;
}

template <class M>
int unit_jac_lu_t(long n, const double* y, const double* T, const double* fT, const double* gamma, const double* b,
                  double* J, double* x, double* keep, int* sing) {
  constexpr int N1 = M::N1;
  const long nw = (n + 63) / 64;
  double *dy = dev_copy(y, n * N1), *dT = dev_copy(T, n), *dfT = dev_copy(fT, n), *dg = dev_copy(gamma, n);
  double *db = dev_copy(b, n * N1), *dJ = dev_zero<double>(n * N1 * N1), *dx = dev_zero<double>(n * N1);
  double* dk = dev_zero<double>(n * N1 + 4 * n);
  int* ds = dev_zero<int>(n);
  double* ws = dev_zero<double>(nw * Slots<N1>::TOTAL * 64);
  double* iws = dev_zero<double>(nw * 64 * MatSlots<N1>::STRIDE);
  hipLaunchKernelGGL(k_jac_lu<M>, dim3((unsigned)nw), dim3(64), 0, nullptr, dy, dT, dfT, dg, db, dJ, dx, dk, ds, ws,
                     iws, n);
  UNIT_SYNC();
  UNIT_D2H(J, dJ, n * N1 * N1 * sizeof(double));
  UNIT_D2H(x, dx, n * N1 * sizeof(double));
  UNIT_D2H(keep, dk, (n * N1 + 4 * n) * sizeof(double));
  UNIT_D2H(sing, ds, n * sizeof(int));
  for (void* p : {(void*)dy, (void*)dT, (void*)dfT, (void*)dg, (void*)db, (void*)dJ, (void*)dx, (void*)dk, (void*)ds,
                  (void*)ws, (void*)iws})
    UNIT_DEV_FREE(p);
  return 0;
}

template <class M>
int unit_coeffs_t(long n, const double* scal, const double* zn, double* out) {
  constexpr int N1 = M::N1;
  const long nw = (n + 63) / 64;
  const long no = n * (14 + 12 * N1);
  double *ds = dev_copy(scal, n * 13), *dz = dev_copy(zn, n * LMAX * N1), *dout = dev_zero<double>(no);
  double* ws = dev_zero<double>(nw * Slots<N1>::TOTAL * 64);
  hipLaunchKernelGGL(k_coeffs<M>, dim3((unsigned)nw), dim3(64), 0, nullptr, ds, dz, dout, ws, n);
  UNIT_SYNC();
  UNIT_D2H(out, dout, no * sizeof(double));
  for (void* p : {(void*)ds, (void*)dz, (void*)dout, (void*)ws}) UNIT_DEV_FREE(p);
  return 0;
}


// Step-size / order control of one lane after a successful step (prepare_next_step,
// including pow-based eta estimates) and after a failed error test's first retry.
// scal in : [q, qmax, qwait, etamax, h, dsm, tq1..tq5, saved_tq5, tau1..tau6]  (18)
// vectors : zn (LMAX*N1), acor (N1), ewt (N1)
// out     : [eta, qprime, hprime, qwait, zn[qmax] after (N1)], then pow(x, y) table
template <class M>
__global__ void k_stepctl(const double* scal, const double* zn_in, const double* acor, const double* ewt,
                          double* out, const double* px, const double* py, double* pz, double* ws, long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  Lane<M> st;
  st.ws.p = ws + (c >> 6) * (long)S::TOTAL * 64 + (c & 63);
  const double* s = scal + c * 18;
  st.q = (int)s[0];
  st.qmax = (int)s[1];
  st.qwait = (int)s[2];
  st.etamax = s[3];
  st.h = s[4];
  st.dsm = s[5];
  st.tq[0] = 0.0;
  for (int i = 1; i <= 5; ++i) st.tq[i] = s[5 + i];
  st.saved_tq5 = s[11];
  st.tau[0] = 0.0;
  for (int i = 1; i <= LMAX; ++i) st.tau[i] = s[11 + i];
  st.L = st.q + 1;
  st.eta = -1.0;
  st.qprime = -1;
  st.hprime = -1.0;
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) st.zn(j, i) = zn_in[(c * LMAX + j) * N1 + i];
  for (int i = 0; i < N1; ++i) {
    st.ws[S::ACOR + i] = acor[c * N1 + i];
    st.ws[S::EWT + i] = ewt[c * N1 + i];
  }
  st.prepare_next_step();
  double* o = out + c * (4 + N1);
  o[0] = st.eta;
  o[1] = (double)st.qprime;
  o[2] = st.hprime;
  o[3] = (double)st.qwait;
  for (int i = 0; i < N1; ++i) o[4 + i] = st.zn(st.qmax, i);
  pz[c] = pow(px[c], py[c]);
}

template <class M>
int unit_stepctl_t(long n, const double* scal, const double* zn, const double* acor, const double* ewt, double* out,
                   const double* px, const double* py, double* pz) {
  constexpr int N1 = M::N1;
  const long nw = (n + 63) / 64;
  double *ds = dev_copy(scal, n * 18), *dz = dev_copy(zn, n * LMAX * N1), *da = dev_copy(acor, n * N1);
  double *de = dev_copy(ewt, n * N1), *dout = dev_zero<double>(n * (4 + N1));
  double *dpx = dev_copy(px, n), *dpy = dev_copy(py, n), *dpz = dev_zero<double>(n);
  double* ws = dev_zero<double>(nw * Slots<N1>::TOTAL * 64);
  hipLaunchKernelGGL(k_stepctl<M>, dim3((unsigned)nw), dim3(64), 0, nullptr, ds, dz, da, de, dout, dpx, dpy, dpz, ws,
                     n);
  UNIT_SYNC();
  UNIT_D2H(out, dout, n * (4 + N1) * sizeof(double));
  UNIT_D2H(pz, dpz, n * sizeof(double));
  for (void* p : {(void*)ds, (void*)dz, (void*)da, (void*)de, (void*)dout, (void*)dpx, (void*)dpy, (void*)dpz,
                  (void*)ws})
    UNIT_DEV_FREE(p);
  return 0;
}

// LU of I - gamma J and the Newton solve by the reactor's kernels (cooperative or one
// lane per cell, FP64 or FP32 factors with FP64-residual refinement) on given
// matrices.  Cells with pend[c] == 0 have no set-up pending and must be left as they
// were (factor words 7.0, permutation -1, singularity word -3).  The solve runs on the
// pending, non-singular cells with right-hand side b and error weights ewt.
template <class M>
__global__ void k_lu_prep(const double* J, const double* gamma, const int* pend, const double* b, const double* ewt,
                          double* ws, double* mats, long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  using MS = MatSlots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  const WS w = cell_ws<M>(ws, c);
  const CM mat = cell_mat<M>(mats, c);
  Lane<M> st;
  __builtin_memset(&st, 0, sizeof(st));
  st.gamma = gamma[c];
  st.gammap = gamma[c];
  st.setup_pending = pend[c];
  st.phase = PH_NEWTON;
  store_lane(st, w);
  for (int e = 0; e < N1 * N1; ++e) {
    mat[MS::JS + e] = J[c * N1 * N1 + e];
    mat[MS::LU + e] = 7.0;
  }
  for (int i = 0; i < N1; ++i) {
    mat.perm(MS::PERM, i) = -1;
    mat[MS::B + i] = b[c * N1 + i];
    mat[MS::X + i] = 0.0;
    w[S::EWT + i] = ewt[c * N1 + i];
  }
  mat[MS::IRS] = -1.0;
  mat[MS::IRF] = -1.0;
  w[S::SING] = -3.0;
}

template <class M, class Real>
__global__ void k_lu_read(double* x, double* sing, double* lu, int* perm, double* ir, double* ws, double* mats,
                          long ncell) {
  constexpr int N1 = M::N1;
  using S = Slots<N1>;
  using MS = MatSlots<N1>;
  const long c = (long)blockIdx.x * 64 + threadIdx.x;
  if (c >= ncell) return;
  const WS w = cell_ws<M>(ws, c);
  const CM mat = cell_mat<M>(mats, c);
  sing[c] = w[S::SING];
  const bool untouched = (w[S::SING] == -3.0);
  for (int e = 0; e < N1 * N1; ++e)
    lu[c * N1 * N1 + e] = untouched ? mat[MS::LU + e] : (double)LUAcc<N1, Real>::at(mat, e);
  for (int i = 0; i < N1; ++i) {
    perm[c * N1 + i] = mat.perm(MS::PERM, i);
    x[c * N1 + i] = mat[MS::X + i];
  }
  ir[2 * c] = mat[MS::IRS];
  ir[2 * c + 1] = mat[MS::IRF];
}

#ifndef UNIT_HOST
// one 16 x 16 x 4 matrix-core product on raw lane registers: lane l passes a[l], b[l]
// and c[4 l + v] (v = 0..3) and returns its four result registers in d[4 l + v]
template <class Real>
__global__ void __launch_bounds__(64) k_mfma_probe(const double* a, const double* b, const double* c, double* d) {
  const int l = threadIdx.x;
  typename MatCore<Real>::V4 cv;
  for (int v = 0; v < 4; ++v) cv[v] = (Real)c[4 * l + v];
  cv = MatCore<Real>::mac((Real)a[l], (Real)b[l], cv);
  for (int v = 0; v < 4; ++v) d[4 * l + v] = (double)cv[v];
}

// the pivot searches' group maximum on raw lane keys: lane l passes key[l] and returns
// the maximum over its half-wave (out[l]) and over the wave (out[64 + l])
__global__ void __launch_bounds__(64) k_group_max(const unsigned long long* key, unsigned long long* out) {
  const int l = threadIdx.x;
  out[l] = group_max_u64<32>(key[l]);
  out[64 + l] = group_max_u64<64>(key[l]);
}

// one v_mfma_f32_16x16x32_bf16 on raw lane registers: lane l passes a[8 l + i], b[8 l + i]
// (i = 0..7, values exactly representable in bf16) and c[4 l + v], and returns d[4 l + v]
typedef __bf16 unit_bf16x8 __attribute__((ext_vector_type(8)));
__global__ void __launch_bounds__(64) k_mfma_bf16_probe(const float* a, const float* b, const float* c, float* d) {
  const int l = threadIdx.x;
  unit_bf16x8 av, bv;
  for (int i = 0; i < 8; ++i) {
    av[i] = (__bf16)a[8 * l + i];
    bv[i] = (__bf16)b[8 * l + i];
  }
  typedef float v4 __attribute__((ext_vector_type(4)));
  v4 cv;
  for (int v = 0; v < 4; ++v) cv[v] = c[4 * l + v];
  cv = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, cv, 0, 0, 0);
  for (int v = 0; v < 4; ++v) d[4 * l + v] = cv[v];
}
#endif

template <class M>
int unit_lu_t(int coop, int fp32, int sweeps, long n, const double* J, const double* gamma, const int* pend,
              const double* b, const double* ewt, double* x, double* sing, double* lu, int* perm, double* ir) {
  constexpr int N1 = M::N1;
#ifdef UNIT_HOST
  if (coop) return -2;   // lanes of the cooperative kernels cannot run one at a time
#endif
  // coop: 0 one lane per cell, 1 the cooperative LU, 2 the blocked LU on the matrix cores,
  // 3 the cooperative LU that solves its first system itself (the solve kernel does not run)
  const long nw = (n + 63) / 64;
  double *dJ = dev_copy(J, n * N1 * N1), *dg = dev_copy(gamma, n), *db = dev_copy(b, n * N1);
  double* de = dev_copy(ewt, n * N1);
  int* dp = dev_copy(pend, n);
  double *dx = dev_zero<double>(n * N1), *ds = dev_zero<double>(n), *dlu = dev_zero<double>(n * N1 * N1);
  double* dir = dev_zero<double>(2 * n);
  int* dperm = dev_zero<int>(n * N1);
  double* ws = dev_zero<double>(nw * Slots<N1>::TOTAL * 64);
  int* iws = dev_zero<int>(nw * Slots<N1>::ITOTAL * 64);
  double* mats = dev_zero<double>(nw * 64 * MatSlots<N1>::STRIDE);
  std::vector<int> ident(n);
  for (long i = 0; i < n; ++i) ident[i] = (int)i;
  int* dlist = dev_copy(ident.data(), n);
  unsigned int hcounts[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  unsigned int* dcount = dev_copy(hcounts, 8);
  ReactArgs a;
  __builtin_memset(&a, 0, sizeof(a));
  a.ws = ws;
  a.iws = iws;
  a.mat = mats;
  a.counts = dcount;
  a.lu_mode = fp32 ? LU_FP32_IR : LU_FP64;
  a.ir_sweeps = sweeps;
  a.ir_tol = 1e-4;
  a.lu_lane = coop ? 0 : 1;
  a.lu_mfma = coop == 2 ? 1 : 0;
  a.fuse = coop == 3 ? 1 : 0;
  hipLaunchKernelGGL(k_lu_prep<M>, dim3((unsigned)nw), dim3(64), 0, nullptr, dJ, dg, dp, db, de, ws, mats, n);
  hcounts[0] = (unsigned)n;
  UNIT_H2D(dcount, hcounts, sizeof(hcounts));
  (void)launch_lu<M>(a, dlist, &dcount[0], n, nullptr);
  UNIT_SYNC();
  // solve list: pending cells whose factorisation is regular (solve_due skips the rest)
  std::vector<double> hs(n);
  if (fp32)
    hipLaunchKernelGGL((k_lu_read<M, float>), dim3((unsigned)nw), dim3(64), 0, nullptr, dx, ds, dlu, dperm, dir, ws,
                       mats, n);
  else
    hipLaunchKernelGGL((k_lu_read<M, double>), dim3((unsigned)nw), dim3(64), 0, nullptr, dx, ds, dlu, dperm, dir, ws,
                       mats, n);
  UNIT_SYNC();
  UNIT_D2H(hs.data(), ds, n * sizeof(double));
  std::vector<int> sl;
  for (long i = 0; i < n; ++i)
    if (pend[i] && hs[i] == 0.0 && coop != 3) sl.push_back((int)i);
  int* dsl = dev_copy(sl.empty() ? ident.data() : sl.data(), sl.empty() ? 1 : (long)sl.size());
  hcounts[6] = (unsigned)sl.size();
  UNIT_H2D(dcount, hcounts, sizeof(hcounts));
  a.nlist = dsl;
  if (!sl.empty()) (void)launch_solve<M>(a, (long)sl.size(), nullptr);
  if (fp32)
    hipLaunchKernelGGL((k_lu_read<M, float>), dim3((unsigned)nw), dim3(64), 0, nullptr, dx, ds, dlu, dperm, dir, ws,
                       mats, n);
  else
    hipLaunchKernelGGL((k_lu_read<M, double>), dim3((unsigned)nw), dim3(64), 0, nullptr, dx, ds, dlu, dperm, dir, ws,
                       mats, n);
  UNIT_SYNC();
  UNIT_D2H(x, dx, n * N1 * sizeof(double));
  UNIT_D2H(sing, ds, n * sizeof(double));
  UNIT_D2H(lu, dlu, n * N1 * N1 * sizeof(double));
  UNIT_D2H(perm, dperm, n * N1 * sizeof(int));
  UNIT_D2H(ir, dir, 2 * n * sizeof(double));
  for (void* p : {(void*)dJ, (void*)dg, (void*)db, (void*)de, (void*)dp, (void*)dx, (void*)ds, (void*)dlu,
                  (void*)dir, (void*)dperm, (void*)ws, (void*)iws, (void*)mats, (void*)dlist, (void*)dcount,
                  (void*)dsl})
    UNIT_DEV_FREE(p);
  return 0;
}
}  // namespace
}  // namespace pelelm

using namespace pelelm;

extern "C" int unit_lu(const char* mech, int coop, int fp32, int sweeps, long n, const double* J, const double* gamma,
                       const int* pend, const double* b, const double* ewt, double* x, double* sing, double* lu,
                       int* perm, double* ir) {
  const int m = mech_lookup(mech);
  if (m == MECH_DRM19) return unit_lu_t<mech_drm19>(coop, fp32, sweeps, n, J, gamma, pend, b, ewt, x, sing, lu, perm, ir);
  if (m == MECH_DODECANE53) return unit_lu_t<mech_dodecane53>(coop, fp32, sweeps, n, J, gamma, pend, b, ewt, x, sing, lu, perm, ir);
  if (m == MECH_LIDRYER)
    return unit_lu_t<mech_LiDryer>(coop, fp32, sweeps, n, J, gamma, pend, b, ewt, x, sing, lu, perm, ir);
  return -1;
}

// f64: 1 v_mfma_f64_16x16x4_f64, 0 v_mfma_f32_16x16x4_f32 (operands rounded to FP32);
// a, b: 64 lane values, c, d: 256 (lane-major, four registers per lane)
extern "C" int unit_mfma_probe(int f64, const double* A, const double* B, const double* Cm, double* D) {
#ifdef UNIT_HOST
  (void)f64; (void)A; (void)B; (void)Cm; (void)D;
  return -2;   // a matrix-core product needs a whole wave
#else
  double *dA = dev_copy(A, 64), *dB = dev_copy(B, 64), *dC = dev_copy(Cm, 256), *dD = dev_zero<double>(256);
  if (f64)
    hipLaunchKernelGGL(k_mfma_probe<double>, dim3(1), dim3(64), 0, nullptr, dA, dB, dC, dD);
  else
    hipLaunchKernelGGL(k_mfma_probe<float>, dim3(1), dim3(64), 0, nullptr, dA, dB, dC, dD);
  const hipError_t e = hipGetLastError();
  UNIT_SYNC();
  UNIT_D2H(D, dD, 256 * sizeof(double));
  for (double* p : {dA, dB, dC, dD}) UNIT_DEV_FREE(p);
  return e == hipSuccess ? 0 : -3;
#endif
}

// key: 64 lane keys; out: 128 (half-wave maxima, then wave maxima)
extern "C" int unit_group_max(const unsigned long long* key, unsigned long long* out) {
#ifdef UNIT_HOST
  (void)key; (void)out;
  return -2;   // a DPP maximum needs a whole wave
#else
  unsigned long long *dk = dev_copy(key, 64), *dout = dev_zero<unsigned long long>(128);
  hipLaunchKernelGGL(k_group_max, dim3(1), dim3(64), 0, nullptr, dk, dout);
  const hipError_t e = hipGetLastError();
  UNIT_SYNC();
  UNIT_D2H(out, dout, 128 * sizeof(unsigned long long));
  for (unsigned long long* p : {dk, dout}) UNIT_DEV_FREE(p);
  return e == hipSuccess ? 0 : -3;
#endif
}

// a, b: 512 lane values (eight per lane), c, d: 256 (four per lane)
extern "C" int unit_mfma_bf16_probe(const float* A, const float* B, const float* Cm, float* D) {
#ifdef UNIT_HOST
  (void)A; (void)B; (void)Cm; (void)D;
  return -2;
#else
  float *dA = dev_copy(A, 512), *dB = dev_copy(B, 512), *dC = dev_copy(Cm, 256), *dD = dev_zero<float>(256);
  hipLaunchKernelGGL(k_mfma_bf16_probe, dim3(1), dim3(64), 0, nullptr, dA, dB, dC, dD);
  const hipError_t e = hipGetLastError();
  UNIT_SYNC();
  UNIT_D2H(D, dD, 256 * sizeof(float));
  for (float* p : {dA, dB, dC, dD}) UNIT_DEV_FREE(p);
  return e == hipSuccess ? 0 : -3;
#endif
}

extern "C" int unit_rhs(const char* mech, long n, const double* y, const double* t, const double* rE0,
                        const double* fH, const double* fy, double* f, double* T) {
  const int m = mech_lookup(mech);
  if (m == MECH_DRM19) return unit_rhs_t<mech_drm19>(n, y, t, rE0, fH, fy, f, T);
  if (m == MECH_DODECANE53) return unit_rhs_t<mech_dodecane53>(n, y, t, rE0, fH, fy, f, T);
  if (m == MECH_LIDRYER) return unit_rhs_t<mech_LiDryer>(n, y, t, rE0, fH, fy, f, T);
  return -1;
}
extern "C" int unit_jac_lu(const char* mech, long n, const double* y, const double* T, const double* fT,
                           const double* gamma, const double* b, double* J, double* x, double* keep, int* sing) {
  const int m = mech_lookup(mech);
  if (m == MECH_DRM19) return unit_jac_lu_t<mech_drm19>(n, y, T, fT, gamma, b, J, x, keep, sing);
  if (m == MECH_DODECANE53) return unit_jac_lu_t<mech_dodecane53>(n, y, T, fT, gamma, b, J, x, keep, sing);
  if (m == MECH_LIDRYER) return unit_jac_lu_t<mech_LiDryer>(n, y, T, fT, gamma, b, J, x, keep, sing);
  return -1;
}
extern "C" int unit_coeffs(const char* mech, long n, const double* scal, const double* zn, double* out) {
  const int m = mech_lookup(mech);
  if (m == MECH_DRM19) return unit_coeffs_t<mech_drm19>(n, scal, zn, out);
  if (m == MECH_DODECANE53) return unit_coeffs_t<mech_dodecane53>(n, scal, zn, out);
  if (m == MECH_LIDRYER) return unit_coeffs_t<mech_LiDryer>(n, scal, zn, out);
  return -1;
}
extern "C" int unit_stepctl(const char* mech, long n, const double* scal, const double* zn, const double* acor,
                            const double* ewt, double* out, const double* px, const double* py, double* pz) {
  const int m = mech_lookup(mech);
  if (m == MECH_DRM19) return unit_stepctl_t<mech_drm19>(n, scal, zn, acor, ewt, out, px, py, pz);
  if (m == MECH_DODECANE53) return unit_stepctl_t<mech_dodecane53>(n, scal, zn, acor, ewt, out, px, py, pz);
  if (m == MECH_LIDRYER) return unit_stepctl_t<mech_LiDryer>(n, scal, zn, acor, ewt, out, px, py, pz);
  return -1;
}
