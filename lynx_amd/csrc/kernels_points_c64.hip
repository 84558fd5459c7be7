// The one-point-per-thread stencil step for float2 elements.
#include "stencil_points.hpp"

LYNX_POINTS(float2, c64)
