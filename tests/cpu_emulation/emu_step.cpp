// One trip of a cell's step logic (Lane::newton_begin, newton_add, trip_end) from a given
// state, on the CPU.  Scalars travel by name order: the lists below and in the test.
#define PELE_WAVES_PER_EU(n)
#include <limits>
#include <vector>

#include "../../pelelm_amd/csrc/reactor_bdf.hip"

thread_local Idx3 threadIdx, blockIdx, blockDim, gridDim;

using namespace pelelm;
using Mech = PELE_TU_MECH_TYPE;

extern "C" int step_n1() { return Mech::N1; }

// d: tn h hprime hscale eta etamax gamma gammap gamrat rl1 crate delp saved_tq5 saved_t a1 a2
//    teval rtol tout, tq[6], l[6], tau[7]
// n: q qprime L qwait nst nstlp nstlj nstloc ncf nef nflag m convfail phase status
//    setup_pending jcur callSetup qmax mxstep
// vectors: zn[6][N1], ewt, acor, x (the Newton solution), f, atol; returns 1 when tout is reached
extern "C" int step_trip(double* d, int* n, double* zn, double* ewt, double* acor, const double* x, const double* f,
                         const double* atol, int singular, int* finite_out) {
  constexpr int N1 = Mech::N1;
  using S = Slots<N1>;
  // the words of one wave's tile; what the trip does not write or read stays NaN
  std::vector<double> ws((size_t)64 * S::TOTAL, std::numeric_limits<double>::quiet_NaN());
  Lane<Mech> st;
  __builtin_memset(&st, 0, sizeof(st));
  st.ws = cell_ws<Mech>(ws.data(), 0);
  double* scal[] = {&st.tn, &st.h, &st.hprime, &st.hscale, &st.eta, &st.etamax, &st.gamma, &st.gammap, &st.gamrat,
                    &st.rl1, &st.crate, &st.delp, &st.saved_tq5, &st.saved_t, &st.a1, &st.a2, &st.teval, &st.rtol,
                    &st.tout};
  int* ints[] = {&st.q, &st.qprime, &st.L, &st.qwait, &st.nst, &st.nstlp, &st.nstlj, &st.nstloc, &st.ncf, &st.nef,
                 &st.nflag, &st.m, &st.convfail, &st.phase, &st.status, &st.setup_pending};
  int at = 0;
  for (double* p : scal) *p = d[at++];
  for (int i = 0; i < 6; ++i) st.tq[i] = d[at++];
  for (int i = 0; i < LMAX; ++i) st.l[i] = d[at++];
  for (int i = 0; i <= LMAX; ++i) st.tau[i] = d[at++];
  at = 0;
  for (int* p : ints) *p = n[at++];
  st.jcur = n[at++] != 0;
  st.callSetup = n[at++] != 0;
  st.qmax = n[at++];
  st.mxstep = n[at++];
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) st.zn(j, i) = zn[j * N1 + i];
  for (int i = 0; i < N1; ++i) {
    st.ws[S::EWT + i] = ewt[i];
    if (st.a2 != 0.0) st.ws[S::ACOR + i] = acor[i];   // not read while the correction is zero
    st.ws[S::F + i] = f[i];
  }
  ReactArgs a{};
  a.rtol = st.rtol;
  for (int i = 0; i < N1; ++i) a.atol[i] = atol[i];
  Lane<Mech>::Newton nw;
  st.newton_begin(nw, singular);
  if (nw.on)
    for (int i = 0; i < N1; ++i) st.newton_add(nw, i, x[i]);
  bool finite = true;
  const bool reached = st.trip_end(a, nw, finite);
  at = 0;
  for (double* p : scal) d[at++] = *p;
  for (int i = 0; i < 6; ++i) d[at++] = st.tq[i];
  for (int i = 0; i < LMAX; ++i) d[at++] = st.l[i];
  for (int i = 0; i <= LMAX; ++i) d[at++] = st.tau[i];
  at = 0;
  for (int* p : ints) n[at++] = *p;
  n[at++] = st.jcur;
  n[at++] = st.callSetup;
  for (int j = 0; j < LMAX; ++j)
    for (int i = 0; i < N1; ++i) zn[j * N1 + i] = st.zn(j, i);
  for (int i = 0; i < N1; ++i) {
    ewt[i] = st.ws[S::EWT + i];
    acor[i] = st.ws[S::ACOR + i];
  }
  *finite_out = finite ? 1 : 0;
  return reached ? 1 : 0;
}
