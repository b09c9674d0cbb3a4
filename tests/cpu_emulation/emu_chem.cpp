// Production rates and the Jacobian of one mechanism (PELE_TU_MECH and its companions on
// the compiler's command line), run serially on the CPU.
#define PELE_WAVES_PER_EU(n)
#include <limits>
#include <vector>

#include "../../pelelm_amd/csrc/reactor_bdf.hip"

thread_local Idx3 threadIdx, blockIdx, blockDim, gridDim;

using namespace pelelm;
using Mech = PELE_TU_MECH_TYPE;

// rates of flat cells (CGS), T re-solved from the enthalpy in place
extern "C" int chem_rates(long n, const double* rY, const double* rH, double* T, double* out) {
  RatesArgs ra{};
  ra.rhoY.p = const_cast<double*>(rY); ra.rhoY.ns = n;
  ra.rhoH.p = const_cast<double*>(rH); ra.rhoH.ns = n;
  ra.T.p = T; ra.T.ns = n;
  ra.rdot.p = out; ra.rdot.ns = n;

  ra.Tout = T;
  ra.nx = (int)n;
  ra.ncell = n;
  return (int)PELE_TU_MECH_FN()->launch_rates(ra, nullptr);
}

// Jacobian (row-major, N1 x N1) of n cells y[n][N1] (rhoY, T) without forcing, fT = dT/dt
extern "C" void chem_jac(long n, const double* y, const double* fT, double* J) {
  constexpr int N1 = Mech::N1;
  using S = Slots<N1>;
  std::vector<double> ws((size_t)((n + 63) / 64) * 64 * S::TOTAL, std::numeric_limits<double>::quiet_NaN());
  for (long c = 0; c < n; ++c) {
    const WS w = cell_ws<Mech>(ws.data(), c);
    for (int k = 0; k < N1 - 1; ++k) w[S::FY + k] = 0.0;
    jacobian<Mech>(y + c * N1, y[c * N1 + N1 - 1], fT[c], w);
    for (int e = 0; e < N1 * N1; ++e) J[c * N1 * N1 + e] = w[S::JS + e];
  }
}

extern "C" void chem_range(double* low, double* high) {
  *low = Mech::T_LOW;
  *high = Mech::T_HIGH;
}
