// cells.hpp -- the cell of a position, as every ordering by cell computes it: the
// list builds take an atom's stencil from the cell that the ordering gave it and
// its wrapped copy from the same fraction, so all of them have to round alike.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace parm {

// Cell of x, x fastest; frac: x in units of the box edges, wrapped into [0, 1).
template <int D>
__device__ __forceinline__ uint32_t cell_of(const Vec<D> &x, const CellGrid &g, Vec<D> &frac) {
    uint32_t key = 0;
#pragma unroll
    for (int k = D - 1; k >= 0; k--) {
        double s = x.c[k] * g.invL[k];
        s -= floor(s);
        frac.c[k] = s;
        int c = (int)(s * (double)g.nc[k]);
        c = c < 0 ? 0 : (c >= g.nc[k] ? g.nc[k] - 1 : c);
        key = key * (uint32_t)g.nc[k] + (uint32_t)c;
    }
    return key;
}

template <int D>
__device__ __forceinline__ uint32_t cell_of(const Vec<D> &x, const CellGrid &g) {
    Vec<D> frac;
    return cell_of<D>(x, g, frac);
}

// x wrapped into [0, L) per component.
template <int D>
__device__ __forceinline__ Vec<D> wrapped(const Vec<D> &x, const CellGrid &g, const Box &box) {
    Vec<D> w;
    (void)cell_of<D>(x, g, w);
#pragma unroll
    for (int k = 0; k < D; k++) w.c[k] = w.c[k] * box.L[k];
    return w;
}

}  // namespace parm
