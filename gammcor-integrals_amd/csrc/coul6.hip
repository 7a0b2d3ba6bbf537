// Hermite potential kernels of bra order 6.
#include "coul_launch.h"

namespace gi {

CoulFn coul_row6(int F) { return coul_row<6>(F); }

}  // namespace gi
