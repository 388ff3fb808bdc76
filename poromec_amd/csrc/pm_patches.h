// pm_patches.h -- host geometry of parallelepiped meshes (pm_patches.cpp).
#pragma once
#include <vector>

// true if the element with the 1-based vertices v[0..7] and the coordinates x
// (3 a node) is a parallelepiped to the rounding of its coordinates
bool pm_is_parallelepiped(const int *v, const double *x);

// ord: element of every slot; ps: first slot of every patch of up to L
// neighbouring elements.  ix: (numel, 21) 1-based nodes, id: (nnode, 4)
// equations from 1, 0 where restrained
void pm_element_patches(int numel, int nen, int nnodev, const int *ix, const int *id,
                        const double *x, int L, std::vector<int> &ord, std::vector<int> &ps);
