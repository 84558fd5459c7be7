// The one-point-per-thread stencil step for double elements.
#include "stencil_points.hpp"

LYNX_POINTS(double, f64)
