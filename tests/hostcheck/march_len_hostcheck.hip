// Test-only host build of the marching kernel's segment length rule (march_len
// in famrdp-jax_amd/csrc/famrdp_march_geom.h).  Compiled with
// --cuda-host-only; never loaded by the product.
#include <cstdint>

#include "famrdp_march_geom.h"

extern "C" int len_of(int tj, int tk, int L, int nblocks, const int32_t* dims, int slots, double* units, int64_t* wgs) {
  return famrdp::march_len(tj, tk, L, nblocks, dims, slots, units, wgs);
}
