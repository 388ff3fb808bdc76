// pm_affine.h -- element products of parallelepiped elements (pm_affine.hip).
#pragma once
#include "pm_elemargs.h"

// Device data of a mesh whose elements are all parallelepipeds (constant
// Jacobian).  Elements are kept in slots (ord), a patch of up to 64 / lpe
// neighbours after the other.
struct PmAffine {
  int numel = 0, nen = 0, nrn = 0;
  int *ord = nullptr;            // (numel) element of each slot
  int lpe = 4;                   // lanes an element: 64 / lpe elements a patch
  int npatch = 0, max_nodes = 0; // patches, most nodes in one
  int *ps = nullptr;             // (npatch + 1) first slot of each patch
  unsigned int *pn = nullptr;    // (npatch + 1) first entry of each patch in pw
  unsigned int *pw = nullptr;    // the patches' nodes: first free equation << 4 | free dofs
  unsigned short *loc = nullptr; // (numel, nen) patch node of each element node
  unsigned int *en = nullptr;    // (numel, nen) free-dof words of the element nodes
  int mstride = 0;
  unsigned int *minc = nullptr;  // (nrn, mstride) elements at each row block: slot << 5 | node
  int stride = 0;                // patch entries kept per row block (the most any has, to 4)
  unsigned int *gnode = nullptr; // (nrn) the block's first row << 4 | free dofs
  unsigned int *gsrc = nullptr;  // (nrn, stride) offsets of its entries in ye, then `zero`
  unsigned int zero = 0;         // offset of four zeros in ye
  double *ec_op = nullptr;       // (numel, 16) coefficients of the assembled matrix
  double *ec = nullptr;          // (numel, 16) coefficients of one element loop
  double *ye = nullptr;          // patch vectors, 4 values a node
  double *tab = nullptr;         // reference integrals of the matrix
  int max_cols = 0;              // widest row block
  // (host) the first and last row block of each patch's nodes, -1: no free node
  std::vector<int> patch_first, patch_last;
  bool op_valid = false;         // ec_op holds the matrix's coefficients
};

void pm_affine_free(PmAffine *a);
// builds the data if every element is a parallelepiped (c->affine stays null
// otherwise, and where memory for it is short)
int pm_affine_setup(pm_ctx *c, const double *x, const PmHostPattern &pat);
// element loop isw 2 or 4 of pform_pm: E.b -= p of every element, face loads
// included; with lhs the matrix, whose coefficients are kept for products
bool pm_affine_loops(const pm_ctx *c, int isw, int lhs);
int pm_affine_pform(pm_ctx *c, const ElemArgs &E, int isw, int lhs, int rhs);

// Krylov products through the elements: true when the matrix in c->A is the
// one whose coefficients are kept and large enough for it to pay
bool pm_affine_product(const pm_ctx *c, int use32);

// the element part of y = A x: patch vectors into ye
void pm_affine_elements(pm_ctx *c, const double *x, const PmScalars *S);

// y = sum of the patch vectors (rows times m with scale_m), with the dots
// y.w and y.y of nv = 0, 1, 2 as workgroup partials; returns the grid
int pm_affine_gather(pm_ctx *c, double *y, const double *w, const double *m, int nv, bool scale_m,
                     const PmScalars *S);
