// The one-point-per-thread stencil step for double2 elements.
#include "stencil_points.hpp"

LYNX_POINTS(double2, c128)
