// Loops unrolled at compile time.
#ifndef DFTGRID_UNROLL_H
#define DFTGRID_UNROLL_H

#include <type_traits>

namespace dg {

// f(B), f(B+1), ..., f(E-1) with compile-time arguments (std::integral_constant).
template <int B, int E, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

}  // namespace dg

#endif
