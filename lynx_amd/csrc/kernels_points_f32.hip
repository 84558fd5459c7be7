// The one-point-per-thread stencil step for float elements.
#include "stencil_points.hpp"

LYNX_POINTS(float, f32)
