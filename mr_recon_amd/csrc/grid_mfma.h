// Gridding phase 1 on the matrix cores (grid_mfma.hip): host-side entry used by the
// dispatch of nufft_kernels.hip.
#pragma once
#include "common.h"

namespace mra {

struct GridMfmaArgs {
  const float2* ksp;
  const float* dcf;    // or null
  const float* wsort;
  const int* lbase;
  const int* perm;
  const Geom* geoms;   // device
  const Item* items;   // device
  int nitems;
  int nbatch;          // largest batch (coil count) among the problems of the launch
  float2* scratch;
  hipStream_t stream;
};

// 2D with 2 <= P <= 8 (tile edges 8, 16, 32) and 3D with 2 <= P <= 7 (tile edge 8).
inline bool grid_mfma_supported(int ndim, int P) { return P >= 2 && ((ndim == 2 && P <= 8) || (ndim == 3 && P <= 7)); }

// Launches the kernel for (ndim, P, tile edge T); the caller checks grid_mfma_supported.
void launch_grid_mfma(int ndim, int P, int T, const GridMfmaArgs& a);

}  // namespace mra
