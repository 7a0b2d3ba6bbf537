// Hermite potential kernels of bra order 7.
#include "coul_launch.h"

namespace gi {

CoulFn coul_row7(int F) { return coul_row<7>(F); }

}  // namespace gi
