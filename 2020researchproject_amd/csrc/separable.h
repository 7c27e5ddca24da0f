// separable.h - direct solves of separable systems: the pressure and momentum of
// a box, the pressure with an immersed body.
#pragma once

#include <vector>

#include "common.h"
#include "solver_kernels.h"

namespace ibm {

// Spectral form of the system (c0 + sum_a T_a) x = b whose 1-D operators T_a
// (after the boundary folds) are symmetric in a scalar product with positive
// weights: T_a = V diag(lam) Vi, Vi V = I. Matrices are row-major, padded with
// zeros to a multiple of 16 on both sides; lam is ascending.
struct SeparableAxis {
    const double *V, *Vi, *lam;
    int n, np;
};
struct SeparableSys {
    SeparableAxis ax[3];
    double c0;   // the operator is c0 + the sum of the three
    int pinned;  // the row of cell (0, 0, 0) is x = b; the problem is otherwise singular
};

struct GreenBox { int lo[3], hi[3]; };  // end exclusive

// Ghost rows of an immersed body (capacitance matrix method). The box's
// operator A holds in every fluid row; a right-hand side mu at the ghost cells
// makes its solution also meet the ghost rows R x = b_g:
//   (R A^-1 E) mu = b_g - R A^-1 b_fluid,  x = A^-1 (b_fluid + E mu).
// A zero row of R (a cell centre on the surface) is x = b.
// look: the box of the ghost cells and their stencil points, cells: that of the
// ghost cells; fluid, ghost: masks of the interior cells, one word per 16 cells
// of a row.
struct SeparableBody {
    const uint8_t *flag;  // F_SOLID: rows x = b, zero ghost rows among them
    GhostRows<double> G;
    const double *inv64;  // inverse of R A^-1 E, row pitch ld; one of the two
    const float *inv32;
    int ld;
    double *t;            // ng: right-hand side of the ghost rows
    const uint16_t *fluid, *ghost;
    GreenBox look, cells;
};

// Host: eigenvalues (ascending) and matrices of one axis from its folded
// coefficients cm, cp, dm, dp (n each); false when the axis has no such form (a
// periodic axis that is not uniform, an extrapolated outlet that couples the
// wrong way).
bool separable_axis(int n, bool periodic, const std::vector<double> coef[4], std::vector<double> &V,
                    std::vector<double> &Vi, std::vector<double> &lam);

// x = A^-1 b (add: x += A^-1 b) up to rounding, all in the padded layout d;
// s1, s2: scratch vectors of that layout, partial: separable_partials doubles
bool separable_fits(const int n[3]);  // the axes fit the kernels' LDS tiles
long separable_partials(const Dims &d);
void launch_separable(hipStream_t st, const Dims &d, const SeparableSys &S, const double *b, double *s1, double *s2,
                      double *x, bool add, double *partial);
// n systems of one shape at once (not pinned): x[c] = A_c^-1 b[c]; s1, s2: n
// scratch vectors each
constexpr int kSepBatch = 3;
struct SeparableBatch {
    SeparableSys S[kSepBatch];
    const double *in[kSepBatch];
    double *out[kSepBatch];
};
void launch_separable_batch(hipStream_t st, const Dims &d, int n, const SeparableSys *S, const double *const *b,
                            double *const *s1, double *const *s2, double *const *x);
// launch_separable with a body (not pinned); s3: a third scratch vector. Solid cells
// get x = b (+= b).
void launch_separable_body(hipStream_t st, const Dims &d, const SeparableSys &S, const SeparableBody &B,
                           const double *b, double *s1, double *s2, double *s3, double *x, bool add);

// Columns of R A^-1 E for the nsrc ghost cells src[c] = {i, j, slot} of plane
// k: out[slot(g) * ld + slot(c)]. loc: 9 per ghost row, the places of its
// stencil points (8, -1: none) and of its cell in the box [lo, hi); h: a
// scratch vector; green: kGreenVecs scratch vectors, each for `per` sources
constexpr int kGreenVecs = 6;
struct GreenScratch { double *v[kGreenVecs]; int per; };
void launch_green_plane(hipStream_t st, const Dims &d, const SeparableSys &S, int k, const int3 *src, int nsrc,
                        const GreenBox &box, const GhostRows<double> &G, const int *loc, double *h,
                        const GreenScratch &green, double *out, long ld);
// *bad = 1 if one of a[0 .. n) is not finite (left alone else)
template <typename T>
void launch_not_finite(hipStream_t st, const T *a, long n, int *bad);

}  // namespace ibm
