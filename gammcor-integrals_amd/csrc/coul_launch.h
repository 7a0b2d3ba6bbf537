// Launch tables of the Hermite potential kernels, one row of ket orders per
// bra order E; the rows are compiled in separate sources (the unrolled kernels
// of the high orders take the compiler seconds each).
#pragma once
#include "coul_kernel.h"
#include "gi_context.h"

namespace gi {

using CoulFn = void (*)(const CoulArgs &, int groups, hipStream_t);

template <int E, int F>
void launch_coul_class(const CoulArgs &a, int groups, hipStream_t s) {
  hipLaunchKernelGGL((k_coul_j<E, F>), dim3((unsigned)((a.nb + 63) / 64), (unsigned)groups), dim3(256), 0,
                     s, a, a.ket, a.dk);
}

template <int E>
CoulFn coul_row(int F) {
  static const CoulFn row[COUL_FMAX + 1] = {&launch_coul_class<E, 0>, &launch_coul_class<E, 1>,
                                            &launch_coul_class<E, 2>, &launch_coul_class<E, 3>,
                                            &launch_coul_class<E, 4>, &launch_coul_class<E, 5>,
                                            &launch_coul_class<E, 6>};
  return row[F];
}

CoulFn coul_row6(int F);   // coul6.hip
CoulFn coul_row7(int F);   // coul7.hip

}  // namespace gi
