// Block arrays between the device layout (component planes of padded rows) and the host's views
// (all components of a cell together).  The boxes pass through a device buffer in the view's
// order, so that a host view is read or written by one contiguous copy per array.
#pragma once
#include "dev_common.h"

// One array's box of cells: `stage` holds ncomp values per cell, cells i fastest.
struct ViewBox {
    double* field;  // element (lo) of component 0
    double* stage;
    long tot;       // component stride of the field
    int ncomp;
    int n0, n1;     // cells along i and j
    int cells;
    int nx, nxy;    // row and plane strides of the field
};

// Bound by the link to the host (about 57 GB/s), not by these passes: a thread moves one cell,
// component by component (one side coalesced, the other whole cache lines per wave).
template <bool UPLOAD>
__global__ void __launch_bounds__(256) k_view(ViewBox v)
{
    const int lin = blockIdx.x * 256 + threadIdx.x;
    if (lin >= v.cells) return;
    const int i = lin % v.n0, r = lin / v.n0;
    const int j = r % v.n1, k = r / v.n1;
    double* f = v.field + i + (long)j * v.nx + (long)k * v.nxy;
    double* s = v.stage + (long)lin * v.ncomp;
    for (int c = 0; c < v.ncomp; c++) {
        if (UPLOAD)
            f[c * v.tot] = s[c];
        else
            s[c] = f[c * v.tot];
    }
}
