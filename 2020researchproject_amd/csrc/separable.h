// separable.h - direct solve of the pressure system of a box without a body.
#pragma once

#include <vector>

#include "common.h"

namespace ibm {

// Spectral form of the system sum_a T_a x = b whose 1-D operators T_a (after
// the boundary folds) are symmetric in the scalar product of the cell widths:
// T_a = V diag(lam) Vi, Vi V = I. Matrices are row-major, padded with zeros to
// a multiple of 16 on both sides; lam is ascending.
struct SeparableAxis {
    const double *V, *Vi, *lam;
    int n, np;
};
struct SeparableSys {
    SeparableAxis ax[3];
    int pinned;  // the row of cell (0, 0, 0) is x = b; the problem is otherwise singular
};

// Host: eigenvalues (ascending) and matrices of one axis from its folded
// coefficients cm, cp, dm, dp (n each) and cell widths; false when the axis
// has no such form (a periodic axis that is not uniform).
bool separable_axis(int n, bool periodic, const std::vector<double> coef[4], const double *width,
                    std::vector<double> &V, std::vector<double> &Vi, std::vector<double> &lam);

// x = A^-1 b (add: x += A^-1 b) up to rounding, all in the padded layout d;
// s1, s2: scratch vectors of that layout, partial: separable_partials doubles
bool separable_fits(const int n[3]);  // the axes fit the kernels' LDS tiles
long separable_partials(const Dims &d);
void launch_separable(hipStream_t st, const Dims &d, const SeparableSys &S, const double *b, double *s1, double *s2,
                      double *x, bool add, double *partial);

}  // namespace ibm
