// Test-only host build of the stage kernels' Roe flux (famrdp_math.h roe_flux2,
// twice the area-weighted flux) and of its reverse (famrdp_adjoint.h), whose
// reciprocals and roots are the host's own here.  Never loaded by the product.
#include "famrdp_adjoint.h"

using namespace famrdp;

extern "C" {

// n samples, sample-major; full: the form of the RHS entry point
void hc_roe_flux2(int n, int full, const double* pl, const double* pr, const double* S, double g, double* F) {
  StageGas gas{};
  gas.gm1 = g - 1.0;
  gas.gm1h = 0.5 * (g - 1.0);
  gas.cg2 = 2.0 * g / (g - 1.0);
  for (int i = 0; i < n; ++i) {
    if (full) roe_flux2<true>(pl + 5 * i, pr + 5 * i, S + 3 * i, gas, F + 5 * i);
    else roe_flux2<false>(pl + 5 * i, pr + 5 * i, S + 3 * i, gas, F + 5 * i);
  }
}

void hc_roe_flux2_vjp(int n, const double* pl, const double* pr, const double* S, double g, const double* f,
                      double* lpl, double* lpr) {
  for (int i = 0; i < n; ++i)
    roe_flux2_vjp(pl + 5 * i, pr + 5 * i, S + 3 * i, 2.0 * g / (g - 1.0), 0.5 * (g - 1.0), f + 5 * i, lpl + 5 * i,
                  lpr + 5 * i);
}
}
