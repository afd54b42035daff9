// The place of an atom among all atoms by their distance from one of them.
#ifndef DFTGRID_ATOM_ORDER_H
#define DFTGRID_ATOM_ORDER_H

#if defined(__HIP__)
#define DG_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define DG_HOST_DEVICE inline
#endif

namespace dg {

// Number of atoms (x, y, z, Z each) that come before atom m by distance from atom a,
// ties by index.  A distance that is not a number counts as infinite: the places of all
// atoms are a permutation of 0..natoms-1 whatever the coordinates hold, so that a table
// filled by place has no gaps.
DG_HOST_DEVICE int distance_place(const double* atoms, int natoms, int a, int m) {
  auto d2 = [&](int k) {
    const double dx = atoms[4 * k] - atoms[4 * a], dy = atoms[4 * k + 1] - atoms[4 * a + 1],
                 dz = atoms[4 * k + 2] - atoms[4 * a + 2];
    // (fused by hand: the compiler may not round two uses of this differently)
    const double d = __builtin_fma(dz, dz, __builtin_fma(dy, dy, dx * dx));
    return d < __builtin_inf() ? d : __builtin_inf();
  };
  const double d = d2(m);
  int place = 0;
  for (int k = 0; k < natoms; ++k) {
    const double x = d2(k);
    place += (x < d || (x == d && k < m)) ? 1 : 0;
  }
  return place;
}

}  // namespace dg

#endif
