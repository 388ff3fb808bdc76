// pm_patches.h -- host geometry of parallelepiped meshes (pm_patches.cpp).
#pragma once

// true if the element with the 1-based vertices v[0..7] and the coordinates x
// (3 a node) is a parallelepiped to the rounding of its coordinates
bool pm_is_parallelepiped(const int *v, const double *x);
