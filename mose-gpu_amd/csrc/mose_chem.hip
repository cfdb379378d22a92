// The chemistry kernels (mose_chem.hpp, mose_radau.hpp) in their own translation unit, with the parity kernels' flags
// (no contraction: the integrators' roundings are the oracle's).
#include <hip/hip_runtime.h>

#include "mose_chem.hpp"
#include "mose_radau.hpp"

namespace mose {

// a persistent grid of 256-lane workgroups of 4 tpw teams, one cell per team at a time
void launch_chem(const ChemDev& M, ChemArgs A, bool radau5, int cus, hipStream_t s) {
  A.tpw = chem_teams(A.ncell, cus, TeamShape<9>::per_wave);
  const long long wgs = (A.ncell + 4 * A.tpw - 1) / (4 * A.tpw);
  const int grid = (int)(wgs < (long long)cus * 8 ? wgs : (long long)cus * 8);
  if (radau5) {
    if (M.two_rounds) k_radau2<9><<<grid, 256, 0, s>>>(M, A);
    else k_radau<9><<<grid, 256, 0, s>>>(M, A);
  } else {
    if (M.two_rounds) k_chem2<9><<<grid, 256, 0, s>>>(M, A);
    else k_chem<9><<<grid, 256, 0, s>>>(M, A);
  }
}

}  // namespace mose
