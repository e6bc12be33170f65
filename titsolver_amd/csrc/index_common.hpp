// Pieces of the cell-index rebuild shared by its large and small forms.
#pragma once

#include "pair_math.hpp"
#include "sph_kernels.hpp"

namespace tit_amd {

// Global cell key of a position x(k) in tank T; positions outside the grid go
// to the border cells.  bad: a coordinate is not a number.
template <int DIM, class F>
__device__ __forceinline__ uint32_t cell_key(const DevTank& T, F&& pos, bool& bad) {
  uint32_t flat = 0;
#pragma unroll
  for (int k = 0; k < DIM; ++k) {
    const double x = pos(k);
    const double f = (x - T.lo[k]) * T.inv_c[k];
    int c;
    if (!(f == f)) {
      bad = true;
      c = 0;
    } else if (f <= 0.0) {
      c = 0;
    } else if (f >= static_cast<double>(T.nc[k] - 1)) {
      c = T.nc[k] - 1;
    } else {
      c = static_cast<int>(f);
    }
    flat = flat * static_cast<uint32_t>(T.nc[k]) + static_cast<uint32_t>(c);
  }
  return T.cell_off + flat;
}

// Cell coordinates (per axis) of particle i's cell in its tank.
template <int DIM>
__device__ __forceinline__ void cell_coords(const BoundaryArgs& A, const DevTank& T, uint32_t i,
                                            int* c) {
  const uint32_t local = A.key[i] - T.cell_off;
  if constexpr (DIM == 2) {
    c[0] = static_cast<int>(local / T.nc[1]);
    c[1] = static_cast<int>(local % T.nc[1]);
  } else {
    const uint32_t q = local / T.nc[2];
    c[2] = static_cast<int>(local % T.nc[2]);
    c[1] = static_cast<int>(q % T.nc[1]);
    c[0] = static_cast<int>(q / T.nc[1]);
  }
}

// The fixed particle's extrapolated state from the Shepard sums S and H.
template <int DIM>
__device__ __forceinline__ void write_fixed(const BoundaryArgs& A, uint32_t i, double S,
                                            double H) {
  const DevParams& P = A.P;
  const double tiny = 6.0554544523933395e-06;  // cbrt(DBL_EPSILON)
  const double Hs = fabs(S) <= tiny ? 0.0 : H / S;
  const double rho_e = eos_density_from_potential(P, Hs);
  A.s.rho[i] = rho_e;
  const double zero[DIM] = {};
  const double m_e = particle_mass(P, A.id[i]);
  write_pair_data<DIM>(P, A.s, i, zero, rho_e, m_e);
  if (A.wall_rho) {
    const uint32_t k = A.id[i] - A.wall_id0;
    A.wall_rho[k] = rho_e;
    A.s.pv[i].z = static_cast<float>(A.wall_mu[k] * m_e / rho_e);  // V_e = m_e / rho_e
  }
#pragma unroll
  for (int d = 0; d < DIM; ++d) A.s.v[d][i] = 0.0;
}

}  // namespace tit_amd
