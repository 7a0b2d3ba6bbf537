// Hermite potential kernels of bra order 0 to 5 and the launch of every class.
#include "coul_launch.h"

namespace gi {

void launch_coul_j(int E, int F, const CoulArgs &a, int groups, hipStream_t s) {
  if (E < 0 || E > COUL_EMAX || F < 0 || F > COUL_FMAX) throw Error{60, "no potential kernel for this class"};
  CoulFn fn = nullptr;
  switch (E) {
    case 0: fn = coul_row<0>(F); break;
    case 1: fn = coul_row<1>(F); break;
    case 2: fn = coul_row<2>(F); break;
    case 3: fn = coul_row<3>(F); break;
    case 4: fn = coul_row<4>(F); break;
    case 5: fn = coul_row<5>(F); break;
    case 6: fn = coul_row6(F); break;
    default: fn = coul_row7(F); break;
  }
  fn(a, groups, s);
}

}  // namespace gi
