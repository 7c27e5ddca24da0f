// separable.hip - direct solve of a separable pressure system (fast
// diagonalisation: Lynch, Rice & Thomas 1964), with an immersed body by the
// capacitance matrix of its ghost rows (Buzbee, Dorr, George & Golub 1971).
//
// Without an immersed body the pressure operator is a sum of three 1-D
// operators, so it is diagonal in the tensor product of their eigenvectors:
// three dense transforms, a division by the sum of the eigenvalues, three
// transforms back. All of it is matrix products, on the FP64 matrix cores, in
// three launches: the x and y transforms of a plane, the z transform with the
// division and its inverse, the y and x transforms back. Each launch reads and
// writes the field once and keeps the intermediate of its two products in LDS.
// Work: 12 n flops per cell (n: mean axis length), at 128^3 3.2 GFLOP, 41 us at
// the chip's FP64 matrix rate. Measured at 128^3: 55, 60 and 47 us (20 TFLOP/s,
// bound by the operand loads of one 16 x 16 tile per wave); at 32^3 4.6, 6.8
// and 4.7 us, the length of a small launch. A BiCGSTAB iteration with two
// multigrid cycles took 420 us at 128^3 and 190 us at 32^3, and there were 10
// and 6 of them per step.
#include "separable.h"

#include <algorithm>
#include <cmath>
#include <numeric>

namespace ibm {

typedef double mfma_acc __attribute__((ext_vector_type(4)));

constexpr int kSepThreads = 256;
constexpr int kSepWaves = kSepThreads / 64;
// LDS row padding: the four lane groups of an operand read, four rows apart,
// then use different banks
constexpr int kSepPad = 4;

// 16 x 16 tile of a product with K = 16 chunks: lane l holds row (of A) or
// column (of B) l % 16, and the elements 16 c + 4 (l / 16) + 0 .. 3 of the
// summed index in chunk c (any order serves as long as A and B agree). Result
// element r of a lane: row 4 r + l / 16, column l % 16.
template <typename FA, typename FB>
__device__ inline mfma_acc sep_tile(int chunks, FA a, FB b) {
    mfma_acc acc = {0, 0, 0, 0};
    const int k0 = 4 * ((threadIdx.x & 63) >> 4);
    double av[4], bv[4], an[4], bn[4];
    a(k0, av);
    b(k0, bv);
    for (int c = 1; c <= chunks; c++) {
        const int kn = 16 * min(c, chunks - 1) + k0;  // the next chunk's operands, in flight during the products
        a(kn, an);
        b(kn, bn);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t], bv[t], acc, 0, 0, 0);
            av[t] = an[t];
            bv[t] = bn[t];
        }
    }
    return acc;
}

__device__ inline void sep_load4(const double *p, double (&v)[4]) {
    const double2 a = *reinterpret_cast<const double2 *>(p), b = *reinterpret_cast<const double2 *>(p + 2);
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

// What the first transform reads of b at a cell: everything, only fluid cells,
// or only ghost cells (the result is then added to y)
enum { SEP_ALL, SEP_FLUID, SEP_GHOST };

// y(l, m, k) = sum_ij Vi_x[l][i] Vi_y[m][j] b(i, j, k) for the l of one block
// of 16 nb and all m: plane k = k0 + blockIdx.y
template <int WHAT>
__global__ void __launch_bounds__(kSepThreads) k_sep_xy(Dims d, SeparableAxis X, SeparableAxis Y, const double *b,
                                                        const uint8_t *flag, double *y, int nb, int k0) {
    extern __shared__ double sep_lds[];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = k0 + blockIdx.y, l0 = blockIdx.x * 16 * nb, pitch = 16 * nb + kSepPad;
    const int mt = Y.np / 16, nt = min(nb, (X.np - l0) / 16);
    for (int w = wave; w < mt * nt; w += kSepWaves) {
        const int j0 = 16 * (w / nt), c0 = 16 * (w % nt);
        const long q0 = cidx(d, 0, min(j0 + ln, d.ny - 1), k);
        const double *vx = X.Vi + (long)(l0 + c0 + ln) * X.np;
        const mfma_acc t = sep_tile(
            X.np / 16,
            [&](int i, double (&v)[4]) {
                sep_load4(b + q0 + i, v);
                unsigned f = 0;
                if (WHAT != SEP_ALL) f = *reinterpret_cast<const unsigned *>(flag + q0 + i);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const unsigned fq = f >> 8 * q & 0xFF;
                    const bool in = WHAT == SEP_ALL || fq == (WHAT == SEP_FLUID ? F_FLUID : F_GHOST);
                    v[q] = in && i + q < d.nx ? v[q] : 0.0;  // not what lies past the row
                }
            },
            [&](int i, double (&v)[4]) { sep_load4(vx + i, v); });
#pragma unroll
        for (int r = 0; r < 4; r++) sep_lds[(j0 + 4 * r + g) * pitch + c0 + ln] = t[r];
    }
    __syncthreads();
    for (int w = wave; w < mt * nt; w += kSepWaves) {
        const int m0 = 16 * (w / nt), c0 = 16 * (w % nt);
        const double *vy = Y.Vi + (long)(m0 + ln) * Y.np;
        const double *col = sep_lds + c0 + ln;
        const mfma_acc t = sep_tile(
            Y.np / 16, [&](int j, double (&v)[4]) { sep_load4(vy + j, v); },
            [&](int j, double (&v)[4]) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = col[(j + q) * pitch];
            });
        const int l = l0 + c0 + ln;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + 4 * r + g;
            if (l >= d.nx || m >= d.ny) continue;
            const long q = cidx(d, l, m, k);
            y[q] = WHAT == SEP_GHOST ? y[q] + t[r] : t[r];
        }
    }
}

// w(l, m, k) = sum_n V_z[k][n] u(l, m, n), u = (sum_k Vi_z[n][k] y(l, m, k)) /
// (lam_l + lam_m + lam_n), for one row m = blockIdx.y and a block of 16 nb l.
// pinned: b is changed at cell (0, 0, 0) so that the singular problem has a
// solution (the other rows do not see that row), by the multiple of its unit
// vector that takes out the zero mode, and the zero mode of the solution is 0;
// partial gets the block's share of the solution at that cell.
// Planes k of the tiles [t0, t1) are written. UNIT: y is a unit vector in z, 1
// in plane ku for every l and m.
template <bool UNIT>
__global__ void __launch_bounds__(kSepThreads) k_sep_z(Dims d, SeparableSys S, const double *y, double *w_out, int nb,
                                                       int t0, int t1, int ku, double *partial) {
    extern __shared__ double sep_lds[];
    __shared__ double first[kSepThreads / 64 + 1];
    const SeparableAxis &Z = S.ax[2];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int m = blockIdx.y, l0 = blockIdx.x * 16 * nb, pitch = 16 * nb + kSepPad;
    const int zt = Z.np / 16, nt = min(nb, (S.ax[0].np - l0) / 16);
    double shift = 0;  // the added multiple of the unit vector
    if (S.pinned) {
        double z = 0;
        for (int k = threadIdx.x; k < d.nz; k += kSepThreads) z += Z.Vi[k] * y[cidx(d, 0, 0, k)];
        for (int o = 32; o > 0; o >>= 1) z += __shfl_down(z, o, 64);
        if ((threadIdx.x & 63) == 0) first[wave] = z;
        __syncthreads();
        z = 0;
        for (int q = 0; q < kSepWaves; q++) z += first[q];
        shift = -z / (S.ax[0].Vi[0] * S.ax[1].Vi[0] * Z.Vi[0]);
    }
    const double lm = S.ax[1].lam[m];
    const double um = S.pinned ? S.ax[1].Vi[(long)m * S.ax[1].np] * shift : 0.0;
    for (int w = wave; w < zt * nt; w += kSepWaves) {
        const int n0 = 16 * (w / nt), c0 = 16 * (w % nt);
        const int l = min(l0 + c0 + ln, d.nx - 1);
        const double *vz = Z.Vi + (long)(n0 + ln) * Z.np, *col = y + cidx(d, l, m, 0);
        mfma_acc t;
        if (UNIT)
            for (int r = 0; r < 4; r++) t[r] = Z.Vi[(long)(n0 + 4 * r + g) * Z.np + ku];
        else t = sep_tile(
            zt, [&](int k, double (&v)[4]) { sep_load4(vz + k, v); },
            [&](int k, double (&v)[4]) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = col[min(k + q, d.nz - 1) * d.sz];
            });
        const double ll = S.ax[0].lam[l] + lm;
        const double ul = S.pinned ? S.ax[0].Vi[(long)l * S.ax[0].np] * um : 0.0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int n = n0 + 4 * r + g;
            double v = 0;
            if (n < d.nz) {
                const double den = ll + Z.lam[n];
                v = den != 0 ? (t[r] + (S.pinned ? ul * Z.Vi[(long)n * Z.np] : 0.0)) / den : 0.0;
            }
            sep_lds[n * pitch + c0 + ln] = v;
        }
    }
    __syncthreads();
    double mine = 0;
    for (int w = wave; w < (t1 - t0) * nt; w += kSepWaves) {
        const int k0 = 16 * (t0 + w / nt), c0 = 16 * (w % nt);
        const double *vz = Z.V + (long)(k0 + ln) * Z.np, *col = sep_lds + c0 + ln;
        const mfma_acc t = sep_tile(
            zt, [&](int n, double (&v)[4]) { sep_load4(vz + n, v); },
            [&](int n, double (&v)[4]) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = col[(n + q) * pitch];
            });
        const int l = l0 + c0 + ln;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int k = k0 + 4 * r + g;
            if (l < d.nx && k < d.nz) w_out[cidx(d, l, m, k)] = t[r];
        }
        if (S.pinned && k0 == 0 && g == 0 && l < d.nx) mine += S.ax[0].V[l] * t[0];
    }
    if (!S.pinned) return;
    mine *= S.ax[1].V[m];
    for (int o = 32; o > 0; o >>= 1) mine += __shfl_down(mine, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) first[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int q = 0; q < kSepWaves; q++) s += first[q];
        partial[blockIdx.x + (long)gridDim.x * m] = s;
    }
}

// x(i, j, k) = or += sum_lm V_x[i][l] V_y[j][m] w(l, m, k) for all i, the rows j
// of a block of 16 nb from tile t0 (of the tiles below t1) and plane k = k0 +
// blockIdx.y. pinned: plus the constant that gives cell (0, 0, 0) its
// right-hand side (np partial sums of its value). flag: solid cells take b.
__global__ void __launch_bounds__(kSepThreads) k_sep_back(Dims d, SeparableAxis X, SeparableAxis Y, const double *w_in,
                                                          double *x, int nb, int t0, int t1, int k0, int add,
                                                          int pinned, const double *b, const uint8_t *flag,
                                                          const double *partial, int np) {
    extern __shared__ double sep_lds[];
    __shared__ double first[kSepThreads / 64];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = k0 + blockIdx.y, j0 = 16 * (t0 + blockIdx.x * nb), pitch = X.np + kSepPad;
    const int xt = X.np / 16, jt = min(nb, t1 - j0 / 16);
    double base = 0;
    if (pinned) {
        double s = 0;
        for (int q = threadIdx.x; q < np; q += kSepThreads) s += partial[q];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if ((threadIdx.x & 63) == 0) first[wave] = s;
    }
    for (int w = wave; w < jt * xt; w += kSepWaves) {
        const int r0 = 16 * (w / xt), c0 = 16 * (w % xt);
        const int l = min(c0 + ln, d.nx - 1);
        const double *vy = Y.V + (long)(j0 + r0 + ln) * Y.np, *col = w_in + cidx(d, l, 0, k);
        const mfma_acc t = sep_tile(
            Y.np / 16, [&](int m, double (&v)[4]) { sep_load4(vy + m, v); },
            [&](int m, double (&v)[4]) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = col[(long)min(m + q, d.ny - 1) * d.sy];
            });
#pragma unroll
        for (int r = 0; r < 4; r++) sep_lds[(r0 + 4 * r + g) * pitch + c0 + ln] = t[r];
    }
    __syncthreads();
    if (pinned) {
        double s = 0;
        for (int q = 0; q < kSepWaves; q++) s += first[q];
        base = b[cidx(d, 0, 0, 0)] - s;
    }
    for (int w = wave; w < jt * xt; w += kSepWaves) {
        const int r0 = 16 * (w / xt), i0 = 16 * (w % xt);
        const double *vx = X.V + (long)(i0 + ln) * X.np, *row = sep_lds + (r0 + ln) * pitch;
        const mfma_acc t = sep_tile(
            xt, [&](int l, double (&v)[4]) { sep_load4(row + l, v); },
            [&](int l, double (&v)[4]) { sep_load4(vx + l, v); });
        const int i = i0 + ln;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = j0 + r0 + 4 * r + g;
            if (i >= d.nx || j >= d.ny) continue;
            const long q = cidx(d, i, j, k);
            const double v = flag && flag[q] == F_SOLID ? b[q] : t[r] + base;
            x[q] = add ? x[q] + v : v;
        }
    }
}

static int sep_pad16(int n) { return (n + 15) / 16 * 16; }

// LDS of a block of nb tiles of 16 beside a padded axis of np (its larger
// layout: np rows of 16 nb, or 16 nb rows of np)
static size_t sep_lds_bytes(int nb, int np) {
    return std::max((size_t)np * (16 * nb + kSepPad), (size_t)16 * nb * (np + kSepPad)) * sizeof(double);
}
constexpr size_t kSepLds = 64 * 1024;

// Tiles of 16 per block along an axis of `tiles` tiles beside `other` blocks
// of the grid: as many as leave a workgroup for every compute unit and fit
// the LDS, up to four (the matrices are then read by fewer workgroups).
static int sep_block(int tiles, int other, int np) {
    for (int nb = 4; nb > 1; nb /= 2)
        if (tiles >= nb && (long)((tiles + nb - 1) / nb) * other >= 256 && sep_lds_bytes(nb, np) <= kSepLds) return nb;
    return 1;
}

bool separable_fits(const int n[3]) {
    return sep_lds_bytes(1, sep_pad16(std::max({n[0], n[1], n[2]}))) <= kSepLds;
}

long separable_partials(const Dims &d) { return (long)(sep_pad16(d.nx) / 16) * d.ny; }

template <int WHAT>
static void sep_xy(hipStream_t st, const Dims &d, const SeparableSys &S, const double *b, const uint8_t *flag,
                   double *y, int k0, int k1) {
    const int xt = S.ax[0].np / 16, nb = sep_block(xt, k1 - k0, S.ax[1].np);
    hipLaunchKernelGGL((k_sep_xy<WHAT>), dim3((xt + nb - 1) / nb, k1 - k0), dim3(kSepThreads),
                       (size_t)S.ax[1].np * (16 * nb + kSepPad) * sizeof(double), st, d, S.ax[0], S.ax[1], b, flag, y,
                       nb, k0);
}

// planes [k0, k1) (whole tiles of 16); returns the number of partial sums
template <bool UNIT>
static int sep_z(hipStream_t st, const Dims &d, const SeparableSys &S, const double *y, double *w, int k0, int k1,
                 int ku, double *partial) {
    const int xt = S.ax[0].np / 16, nb = sep_block(xt, d.ny, S.ax[2].np), g = (xt + nb - 1) / nb;
    hipLaunchKernelGGL((k_sep_z<UNIT>), dim3(g, d.ny), dim3(kSepThreads),
                       (size_t)S.ax[2].np * (16 * nb + kSepPad) * sizeof(double), st, d, S, y, w, nb, k0 / 16,
                       (k1 + 15) / 16, ku, partial);
    return g * d.ny;
}

// rows [j0, j1) (whole tiles of 16) of the planes [k0, k1)
static void sep_back(hipStream_t st, const Dims &d, const SeparableSys &S, const double *w, double *x, int j0, int j1,
                     int k0, int k1, bool add, const double *b, const uint8_t *flag, const double *partial, int np) {
    const int t0 = j0 / 16, t1 = (j1 + 15) / 16, nb = sep_block(t1 - t0, k1 - k0, S.ax[0].np);
    hipLaunchKernelGGL(k_sep_back, dim3((t1 - t0 + nb - 1) / nb, k1 - k0), dim3(kSepThreads),
                       (size_t)16 * nb * (S.ax[0].np + kSepPad) * sizeof(double), st, d, S.ax[0], S.ax[1], w, x, nb,
                       t0, t1, k0, add ? 1 : 0, partial ? S.pinned : 0, b, flag, partial, np);
}

void launch_separable(hipStream_t st, const Dims &d, const SeparableSys &S, const double *b, double *s1, double *s2,
                      double *x, bool add, double *partial) {
    sep_xy<SEP_ALL>(st, d, S, b, nullptr, s1, 0, d.nz);
    const int np = sep_z<false>(st, d, S, s1, s2, 0, d.nz, 0, partial);
    sep_back(st, d, S, s2, x, 0, d.ny, 0, d.nz, add, b, nullptr, partial, np);
}

// ---------------------------------------------------------------------------
// immersed body
// ---------------------------------------------------------------------------
// One solve is two passes of the transforms, the first one's last two limited
// to the planes and rows the ghost rows look at, and one product with the
// inverse of the ghost rows' matrix: 256 x 128 x 128 with 3568 ghost cells
// 0.63 ms, of it 32 us for the product (102 MB); BiCGSTAB with multigrid
// cycles took 7 iterations of 0.95 ms.
// t_g = b_g - (R y)_g
__global__ void k_cap_rhs(GhostRows<double> G, const double *b, const double *y, double *t) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= G.ng) return;
    double a = 0;
    for (int l = 0; l < 8; l++) {
        const long q = G.src[8 * (long)s + l];
        if (q >= 0) a += G.w[8 * (long)s + l] * y[q];
    }
    const long c = G.cell[s];
    t[s] = b[c] - ((1 - G.wself[s]) * y[c] - a);
}

// mu = inv t into the ghost cells of y: a wave per row, bound by reading the
// inverse once
template <typename T>
__global__ void __launch_bounds__(256) k_cap_apply(GhostRows<double> G, const T *inv, int ld, const double *t,
                                                   double *y) {
    const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (s >= G.ng) return;
    const T *row = inv + (long)s * ld;
    double a[4] = {0, 0, 0, 0};
    int c = lane;
    for (; c + 192 < G.ng; c += 256)
#pragma unroll
        for (int q = 0; q < 4; q++) a[q] += (double)row[c + 64 * q] * t[c + 64 * q];
    for (; c < G.ng; c += 64) a[0] += (double)row[c] * t[c];
    double v = (a[0] + a[1]) + (a[2] + a[3]);
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) y[G.cell[s]] = v;
}

void launch_separable_body(hipStream_t st, const Dims &d, const SeparableSys &S, const SeparableBody &B,
                           const double *b, double *s1, double *s2, double *s3, double *x, bool add) {
    // A^-1 b_fluid where the ghost rows look; then the ghost cells' part is
    // added to its transform
    sep_xy<SEP_FLUID>(st, d, S, b, B.flag, s1, 0, d.nz);
    sep_z<false>(st, d, S, s1, s2, B.z0, B.z1, 0, nullptr);
    sep_back(st, d, S, s2, s3, B.y0, B.y1, B.z0, B.z1, false, b, nullptr, nullptr, 0);
    const int ng = B.G.ng;
    hipLaunchKernelGGL(k_cap_rhs, dim3((ng + 63) / 64), dim3(64), 0, st, B.G, b, s3, B.t);
    if (B.inv64)
        hipLaunchKernelGGL((k_cap_apply<double>), dim3((ng + 3) / 4), dim3(256), 0, st, B.G, B.inv64, B.ld, B.t, s3);
    else
        hipLaunchKernelGGL((k_cap_apply<float>), dim3((ng + 3) / 4), dim3(256), 0, st, B.G, B.inv32, B.ld, B.t, s3);
    sep_xy<SEP_GHOST>(st, d, S, s3, B.flag, s1, B.g0, B.g1);
    sep_z<false>(st, d, S, s1, s2, 0, d.nz, 0, nullptr);
    sep_back(st, d, S, s2, x, 0, d.ny, 0, d.nz, add, b, B.flag, nullptr, 0);
}

// A^-1 e_c in the box, for the unit vectors of the ghost cells c = src0 +
// blockIdx.z of one plane: h holds their common z part (k_sep_z<true>), the
// x and y parts scale the last two transforms' matrices. Rows: 16 from y tile
// box.lo[1] / 16 + blockIdx.x, plane box.lo[2] + blockIdx.y.
__global__ void __launch_bounds__(kSepThreads) k_cap_green(Dims d, SeparableAxis X, SeparableAxis Y, const double *h,
                                                           const int3 *src, int src0, GreenBox box,
                                                           GreenScratch out) {
    extern __shared__ double sep_lds[];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = box.lo[2] + blockIdx.y, j0 = 16 * (box.lo[1] / 16 + blockIdx.x), pitch = X.np + kSepPad;
    const int xt = X.np / 16, x0 = box.lo[0] / 16, x1 = (box.hi[0] + 15) / 16;
    const int3 c = src[src0 + blockIdx.z];
    double *fy = sep_lds + 16 * pitch;  // Vi_y[m][j of the source]
    for (int m = threadIdx.x; m < Y.np; m += kSepThreads) fy[m] = Y.Vi[(long)m * Y.np + c.y];
    __syncthreads();
    for (int w = wave; w < xt; w += kSepWaves) {
        const int l = min(16 * w + ln, d.nx - 1);
        const double *vy = Y.V + (long)(j0 + ln) * Y.np, *col = h + cidx(d, l, 0, k);
        const double fx = X.Vi[(long)l * X.np + c.x];
        const mfma_acc t = sep_tile(
            Y.np / 16, [&](int m, double (&v)[4]) { sep_load4(vy + m, v); },
            [&](int m, double (&v)[4]) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = col[(long)min(m + q, d.ny - 1) * d.sy] * fy[m + q];
            });
#pragma unroll
        for (int r = 0; r < 4; r++) sep_lds[(4 * r + g) * pitch + 16 * w + ln] = t[r] * fx;
    }
    __syncthreads();
    const int bx = box.hi[0] - box.lo[0], by = box.hi[1] - box.lo[1], bz = box.hi[2] - box.lo[2];
    double *o = out.v[blockIdx.z / out.per] + (long)(blockIdx.z % out.per) * bx * by * bz
        + (long)(k - box.lo[2]) * bx * by;
    for (int w = x0 + wave; w < x1; w += kSepWaves) {
        const int i = 16 * w + ln;
        const double *vx = X.V + (long)i * X.np, *row = sep_lds + ln * pitch;
        const mfma_acc t = sep_tile(
            xt, [&](int l, double (&v)[4]) { sep_load4(row + l, v); },
            [&](int l, double (&v)[4]) { sep_load4(vx + l, v); });
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = j0 + 4 * r + g;
            if (i >= box.lo[0] && i < box.hi[0] && j >= box.lo[1] && j < box.hi[1])
                o[(long)(j - box.lo[1]) * bx + i - box.lo[0]] = t[r];
        }
    }
}

// the ghost rows of those columns
__global__ void k_cap_rows(GhostRows<double> G, const int *loc, const int3 *src, int src0, long vol, GreenScratch in,
                           double *out, long ld) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
    if (s >= G.ng) return;
    const double *y = in.v[c / in.per] + (c % in.per) * vol;
    double a = 0;
    for (int l = 0; l < 8; l++) {
        const int q = loc[9 * (long)s + l];
        if (q >= 0) a += G.w[8 * (long)s + l] * y[q];
    }
    out[s * ld + src[src0 + c].z] = (1 - G.wself[s]) * y[loc[9 * (long)s + 8]] - a;
}

void launch_green_plane(hipStream_t st, const Dims &d, const SeparableSys &S, int k, const int3 *src, int nsrc,
                        const GreenBox &box, const GhostRows<double> &G, const int *loc, double *h,
                        const GreenScratch &green, double *out, long ld) {
    const long vol = (long)(box.hi[0] - box.lo[0]) * (box.hi[1] - box.lo[1]) * (box.hi[2] - box.lo[2]);
    sep_z<true>(st, d, S, h, h, box.lo[2], box.hi[2], k, nullptr);
    const int jt = (box.hi[1] + 15) / 16 - box.lo[1] / 16, batch = kGreenVecs * green.per;
    for (int c = 0; c < nsrc; c += batch) {
        const int n = std::min(batch, nsrc - c);
        hipLaunchKernelGGL(k_cap_green, dim3(jt, box.hi[2] - box.lo[2], n), dim3(kSepThreads),
                           (16 * (size_t)(S.ax[0].np + kSepPad) + S.ax[1].np) * sizeof(double), st, d, S.ax[0],
                           S.ax[1], h, src, c, box, green);
        hipLaunchKernelGGL(k_cap_rows, dim3((G.ng + 255) / 256, n), dim3(256), 0, st, G, loc, src, c, vol, green, out,
                           ld);
    }
}

// ---------------------------------------------------------------------------
// host: eigenvectors of one axis
// ---------------------------------------------------------------------------
// Symmetric tridiagonal matrix (diagonal d, e[i] between i and i + 1): QR steps
// with Wilkinson's shift (Golub & Van Loan, Matrix Computations, 8.3.4-8.3.5).
// Each rotation is a similarity of two neighbouring rows and columns, also
// applied to the rows of q (the identity at first, at the end the eigenvectors).
static bool tridiagonal_eigen(std::vector<double> &d, std::vector<double> &e, std::vector<double> &q) {
    const int n = (int)d.size();
    q.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) q[(size_t)i * n + i] = 1;
    const auto small = [&](int i) { return std::fabs(e[i]) <= 1e-17 * (std::fabs(d[i]) + std::fabs(d[i + 1])); };
    int steps = 0;
    for (int hi = n - 1; hi > 0;) {
        if (small(hi - 1)) {
            e[--hi] = 0;
            continue;
        }
        if (++steps > 60 * n) return false;
        int lo = hi - 1;
        while (lo > 0 && !small(lo - 1)) lo--;
        const double half = (d[hi - 1] - d[hi]) / 2;
        const double mu = d[hi] - e[hi - 1] * e[hi - 1] / (half + std::copysign(std::hypot(half, e[hi - 1]), half));
        double lead = d[lo] - mu, bulge = e[lo];
        for (int k = lo; k < hi; k++) {
            const double r = std::hypot(lead, bulge);
            const double c = r > 0 ? lead / r : 1, s = r > 0 ? bulge / r : 0;
            if (k > lo) e[k - 1] = r;
            // [c s; -s c] on both sides of [d_k e_k; e_k d_(k+1)]
            const double dk = d[k], ek = e[k], dn = d[k + 1], cross = 2 * c * s * ek;
            d[k] = c * c * dk + s * s * dn + cross;
            d[k + 1] = s * s * dk + c * c * dn - cross;
            e[k] = c * s * (dn - dk) + (c * c - s * s) * ek;
            lead = e[k];
            if (k + 1 < hi) {
                bulge = s * e[k + 1];
                e[k + 1] *= c;
            }
            double *u = &q[(size_t)k * n], *v = u + n;
            for (int z = 0; z < n; z++) {
                const double uz = u[z], vz = v[z];
                u[z] = c * uz + s * vz;
                v[z] = c * vz - s * uz;
            }
        }
    }
    return true;
}

bool separable_axis(int n, bool periodic, const std::vector<double> coef[4], const double *width,
                    std::vector<double> &V, std::vector<double> &Vi, std::vector<double> &lam) {
    const std::vector<double> &cm = coef[0], &cp = coef[1], &dm = coef[2], &dp = coef[3];
    std::vector<double> q, ev;
    if (periodic) {
        // uniform spacing: Fourier modes
        for (int i = 0; i < n; i++)
            if (std::fabs(cm[i] - cm[0]) > 1e-10 * cm[0] || std::fabs(cp[i] - cm[0]) > 1e-10 * cm[0] ||
                std::fabs(width[i] - width[0]) > 1e-10 * width[0])
                return false;
        for (int m = 0; m < n; m++) {
            const int f = (m + 1) / 2;  // 0, 1, 1, 2, 2, ...
            ev.push_back(2 * cm[0] * (1 - std::cos(2 * M_PI * f / n)));
            for (int i = 0; i < n; i++) {
                const double a = 2 * M_PI * (double)((long)f * i % n) / n;
                const double scale = m == 0 || 2 * f == n ? std::sqrt(1.0 / n) : std::sqrt(2.0 / n);
                q.push_back(scale * (m % 2 ? std::cos(a) : m ? std::sin(a) : 1.0));
            }
        }
    } else {
        std::vector<double> e(n, 0.0);
        ev.resize(n);
        for (int i = 0; i < n; i++) ev[i] = dm[i] + dp[i];
        for (int i = 0; i + 1 < n; i++) {
            // width_i cp_i = width_(i+1) cm_(i+1): the operator is symmetric
            const double a = cp[i] * width[i], b = cm[i + 1] * width[i + 1];
            if (std::fabs(a - b) > 1e-9 * std::fabs(a) || !(a > 0)) return false;
            e[i] = -0.5 * (a + b) / std::sqrt(width[i] * width[i + 1]);
        }
        if (!tridiagonal_eigen(ev, e, q)) return false;
    }
    std::vector<int> order(n);
    std::iota(order.begin(), order.end(), 0);
    std::sort(order.begin(), order.end(), [&](int a, int b) { return ev[a] < ev[b]; });
    // rows that all sum to zero: the lowest eigenvalue is 0
    bool zero = true;
    for (int i = 0; i < n; i++) zero &= std::fabs(dm[i] + dp[i] - cm[i] - cp[i]) <= 1e-10 * (cm[i] + cp[i]);
    const int np = sep_pad16(n);
    V.assign((size_t)np * np, 0.0);
    Vi.assign((size_t)np * np, 0.0);
    lam.assign(np, 0.0);
    for (int m = 0; m < n; m++) {
        const double v = ev[order[m]];
        lam[m] = zero && m == 0 ? 0.0 : v;
        for (int i = 0; i < n; i++) {
            const double z = q[(size_t)order[m] * n + i];
            V[(size_t)i * np + m] = z / std::sqrt(width[i]);
            Vi[(size_t)m * np + i] = z * std::sqrt(width[i]);
        }
    }
    return true;
}

}  // namespace ibm
