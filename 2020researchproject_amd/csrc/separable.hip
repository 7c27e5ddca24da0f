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
// the chip's FP64 matrix rate. Measured at 128^3: 32, 34 and 33 us (32 TFLOP/s;
// 55, 60 and 47 us with one tile per wave at a time: bound by the operands'
// way through the L2); at 32^3 4.6, 7.0 and 5.7 us, the length of a small
// launch. A BiCGSTAB iteration with two multigrid cycles took 420 us at 128^3
// and 190 us at 32^3, and there were 10 and 6 of them per step.
#include "separable.h"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <type_traits>

namespace ibm {

typedef double mfma_acc __attribute__((ext_vector_type(4)));

constexpr int kSepThreads = 512;  // at most; 256 where the tiles feed no more waves
constexpr int kSepWaves = kSepThreads / 64;
__device__ inline int sep_waves() { return blockDim.x >> 6; }
// LDS row padding (doubles) of a tile read by columns and by rows: the lane
// groups of an operand read then use different banks
constexpr int kSepPadCol = 8, kSepPadRow = 2;

// MR x NR tiles of 16 x 16 of a product with 16 `chunks` summed elements: lane l
// holds row (of A) or column (of B) l % 16, and of chunk c the elements 16 c +
// sep_k(l, 0 .. 3) (any order serves as long as A and B agree; this one loads
// 64 contiguous bytes of 16 rows at once). a(r, k0, v) and b(s, k0, v) load
// those of row tile r and column tile s. Result element e of a lane: row 4 e +
// l / 16, column l % 16. The operands come through the L2 of the XCD, whose
// rate bounds the large grids: a tile product reads MR + NR operands for MR NR
// products.
__device__ inline int sep_k(int g, int t) { return 2 * g + (t & 1) + 8 * (t >> 1); }

template <int MR, int NR, typename FA, typename FB>
__device__ inline void sep_tiles(int chunks, FA a, FB b, mfma_acc (&acc)[MR][NR]) {
    double av[MR][4], bv[NR][4], an[MR][4], bn[NR][4];
#pragma unroll
    for (int r = 0; r < MR; r++) {
        a(r, 0, av[r]);
#pragma unroll
        for (int s = 0; s < NR; s++) acc[r][s] = {0, 0, 0, 0};
    }
#pragma unroll
    for (int s = 0; s < NR; s++) b(s, 0, bv[s]);
    for (int c = 1; c <= chunks; c++) {
        const int kn = 16 * min(c, chunks - 1);  // the next chunk's operands, in flight during the products
#pragma unroll
        for (int r = 0; r < MR; r++) a(r, kn, an[r]);
#pragma unroll
        for (int s = 0; s < NR; s++) b(s, kn, bn[s]);
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < MR; r++)
#pragma unroll
                for (int s = 0; s < NR; s++)
                    acc[r][s] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[r][t], bv[s][t], acc[r][s], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 4; t++) {
#pragma unroll
            for (int r = 0; r < MR; r++) av[r][t] = an[r][t];
#pragma unroll
            for (int s = 0; s < NR; s++) bv[s][t] = bn[s][t];
        }
    }
}

// four consecutive-in-pairs elements of a row (p: row start + chunk + 2 g)
__device__ inline void sep_row(const double *p, double (&v)[4]) {
    const double2 a = *reinterpret_cast<const double2 *>(p), b = *reinterpret_cast<const double2 *>(p + 8);
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

// Macro tiles of MR x NR over mt x nt tiles, one per wave at a time: f(m, n)
// with m, n the first tile of each; tiles past the end are clamped by the
// operand loads and skipped by the stores
template <int MR, int NR, typename F>
__device__ inline void sep_macro(int mt, int nt, F f) {
    const int gn = (nt + NR - 1) / NR, total = (mt + MR - 1) / MR * gn;
    for (int w = threadIdx.x >> 6; w < total; w += sep_waves()) f(w / gn * MR, w % gn * NR);
}

// Cells that the first transform reads: all, or those of a bit mask (16 cells
// of a row per word); with SEP_ADD the result is added to y
enum { SEP_ALL, SEP_MASK, SEP_ADD };

// y(l, m, k) = sum_ij Vi_x[l][i] Vi_y[m][j] b(i, j, k) for the l of one block
// of 16 nb and all m: plane k = k0 + blockIdx.y; i and j over the tiles
// [i0, i1) and [j0, j1) (b is 0 elsewhere)
template <int WHAT, int MR, int NR>
__global__ void __launch_bounds__(kSepThreads) k_sep_xy(Dims d, SeparableBatch B, const uint16_t *mask, int nb,
                                                        int pitch, int k0, int i0, int i1, int j0, int j1) {
    extern __shared__ double sep_lds[];
    const SeparableAxis &X = B.S[blockIdx.z].ax[0], &Y = B.S[blockIdx.z].ax[1];
    const double *b = B.in[blockIdx.z];
    double *y = B.out[blockIdx.z];
    const int ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = k0 + blockIdx.y, l0 = blockIdx.x * 16 * nb;
    const int jt = j1 - j0, mt = Y.np / 16, nt = min(nb, (X.np - l0) / 16);
    sep_macro<MR, NR>(jt, nt, [&](int m, int n) {
        long q0[MR];
        const double *vx[NR];
        const uint16_t *in[MR];
        for (int r = 0; r < MR; r++) {
            const int j = min(16 * (j0 + m + r) + ln, d.ny - 1);
            q0[r] = cidx(d, 16 * i0 + 2 * g, j, k);
            in[r] = mask + ((long)k * d.ny + j) * (X.np / 16) + i0;
        }
        for (int s = 0; s < NR; s++) vx[s] = X.Vi + (long)(l0 + 16 * min(n + s, nt - 1) + ln) * X.np + 16 * i0 + 2 * g;
        mfma_acc t[MR][NR];
        sep_tiles<MR, NR>(
            i1 - i0,
            [&](int r, int i, double (&v)[4]) {
                sep_row(b + q0[r] + i, v);
                const unsigned f = WHAT != SEP_ALL ? (unsigned)in[r][i >> 4] >> 2 * g : 0;
#pragma unroll
                for (int e = 0; e < 4; e++)  // not what lies past the row, or outside the mask
                    if (WHAT == SEP_ALL ? 16 * i0 + i + sep_k(g, e) >= d.nx : !(f >> sep_k(0, e) & 1)) v[e] = 0.0;
            },
            [&](int s, int i, double (&v)[4]) { sep_row(vx[s] + i, v); }, t);
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int s = 0; s < NR; s++)
                if (m + r < jt && n + s < nt)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        sep_lds[(16 * (m + r) + 4 * e + g) * pitch + 16 * (n + s) + ln] = t[r][s][e];
    });
    __syncthreads();
    sep_macro<MR, NR>(mt, nt, [&](int m, int n) {
        const double *vy[MR], *col[NR];
        for (int r = 0; r < MR; r++) vy[r] = Y.Vi + (long)(16 * min(m + r, mt - 1) + ln) * Y.np + 16 * j0 + 2 * g;
        for (int s = 0; s < NR; s++) col[s] = sep_lds + 16 * min(n + s, nt - 1) + ln;
        mfma_acc t[MR][NR];
        sep_tiles<MR, NR>(
            jt, [&](int r, int j, double (&v)[4]) { sep_row(vy[r] + j, v); },
            [&](int s, int j, double (&v)[4]) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = col[s][(j + sep_k(g, e)) * pitch];
            },
            t);
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int s = 0; s < NR; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int row = 16 * (m + r) + 4 * e + g, l = l0 + 16 * (n + s) + ln;
                    if (n + s >= nt || l >= d.nx || row >= d.ny) continue;
                    const long q = cidx(d, l, row, k);
                    y[q] = WHAT == SEP_ADD ? y[q] + t[r][s][e] : t[r][s][e];
                }
    });
}

// w(l, m, k) = sum_n V_z[k][n] u(l, m, n), u = (sum_k Vi_z[n][k] y(l, m, k)) /
// (c0 + lam_l + lam_m + lam_n), for one row m = blockIdx.y and a block of 16 nb l.
// pinned: b is changed at cell (0, 0, 0) so that the singular problem has a
// solution (the other rows do not see that row), by the multiple of its unit
// vector that takes out the zero mode, and the zero mode of the solution is 0;
// partial gets the block's share of the solution at that cell.
// Planes k of the tiles [t0, t1) are written. UNIT: y is a unit vector in z, 1
// in plane ku for every l and m.
template <bool UNIT, int MR, int NR>
__global__ void __launch_bounds__(kSepThreads) k_sep_z(Dims d, SeparableBatch B, int nb, int pitch, int t0, int t1,
                                                       int ku, double *partial) {
    extern __shared__ double sep_lds[];
    __shared__ double first[kSepWaves];
    const SeparableSys &S = B.S[blockIdx.z];
    const double *y = B.in[blockIdx.z];
    double *w_out = B.out[blockIdx.z];
    const SeparableAxis &Z = S.ax[2];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int m = blockIdx.y, l0 = blockIdx.x * 16 * nb;
    const int zt = Z.np / 16, nt = min(nb, (S.ax[0].np - l0) / 16);
    double shift = 0;  // the added multiple of the unit vector
    if (S.pinned) {
        double z = 0;
        for (int k = threadIdx.x; k < d.nz; k += blockDim.x) z += Z.Vi[k] * y[cidx(d, 0, 0, k)];
        for (int o = 32; o > 0; o >>= 1) z += __shfl_down(z, o, 64);
        if ((threadIdx.x & 63) == 0) first[wave] = z;
        __syncthreads();
        z = 0;
        for (int q = 0; q < sep_waves(); q++) z += first[q];
        shift = -z / (S.ax[0].Vi[0] * S.ax[1].Vi[0] * Z.Vi[0]);
    }
    const double lm = S.c0 + S.ax[1].lam[m];
    const double um = S.pinned ? S.ax[1].Vi[(long)m * S.ax[1].np] * shift : 0.0;
    sep_macro<MR, NR>(zt, nt, [&](int zr, int n) {
        const double *vz[MR], *col[NR];
        for (int r = 0; r < MR; r++) vz[r] = Z.Vi + (long)(16 * min(zr + r, zt - 1) + ln) * Z.np + 2 * g;
        for (int s = 0; s < NR; s++) col[s] = y + cidx(d, min(l0 + 16 * (n + s) + ln, d.nx - 1), m, 0);
        mfma_acc t[MR][NR];
        if constexpr (UNIT) {
            for (int r = 0; r < MR; r++)
                for (int s = 0; s < NR; s++)
                    for (int e = 0; e < 4; e++)
                        t[r][s][e] = Z.Vi[(long)(16 * min(zr + r, zt - 1) + 4 * e + g) * Z.np + ku];
        } else {
            sep_tiles<MR, NR>(
                zt, [&](int r, int k, double (&v)[4]) { sep_row(vz[r] + k, v); },
                [&](int s, int k, double (&v)[4]) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = col[s][min(k + sep_k(g, e), d.nz - 1) * d.sz];
                },
                t);
        }
#pragma unroll
        for (int s = 0; s < NR; s++) {
            const int l = min(l0 + 16 * (n + s) + ln, d.nx - 1);
            const double ll = S.ax[0].lam[l] + lm;
            const double ul = S.pinned ? S.ax[0].Vi[(long)l * S.ax[0].np] * um : 0.0;
#pragma unroll
            for (int r = 0; r < MR; r++)
                if (zr + r < zt && n + s < nt)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int row = 16 * (zr + r) + 4 * e + g;
                        double v = 0;
                        if (row < d.nz) {
                            const double den = ll + Z.lam[row];
                            v = t[r][s][e];
                            if (S.pinned) v += ul * Z.Vi[(long)row * Z.np];
                            v = den != 0 ? v / den : 0.0;
                        }
                        sep_lds[row * pitch + 16 * (n + s) + ln] = v;
                    }
        }
    });
    __syncthreads();
    double mine = 0;
    sep_macro<MR, NR>(t1 - t0, nt, [&](int zr, int n) {
        const double *vz[MR], *col[NR];
        for (int r = 0; r < MR; r++) vz[r] = Z.V + (long)(16 * min(t0 + zr + r, t1 - 1) + ln) * Z.np + 2 * g;
        for (int s = 0; s < NR; s++) col[s] = sep_lds + 16 * min(n + s, nt - 1) + ln;
        mfma_acc t[MR][NR];
        sep_tiles<MR, NR>(
            zt, [&](int r, int k, double (&v)[4]) { sep_row(vz[r] + k, v); },
            [&](int s, int k, double (&v)[4]) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = col[s][(k + sep_k(g, e)) * pitch];
            },
            t);
#pragma unroll
        for (int s = 0; s < NR; s++) {
            const int l = l0 + 16 * (n + s) + ln;
            if (n + s >= nt || l >= d.nx) continue;
#pragma unroll
            for (int r = 0; r < MR; r++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int k = 16 * (t0 + zr + r) + 4 * e + g;
                    if (t0 + zr + r < t1 && k < d.nz) w_out[cidx(d, l, m, k)] = t[r][s][e];
                }
            if (S.pinned && t0 + zr == 0 && g == 0) mine += S.ax[0].V[l] * t[0][s][0];
        }
    });
    if (!S.pinned) return;
    mine *= S.ax[1].V[m];
    for (int o = 32; o > 0; o >>= 1) mine += __shfl_down(mine, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) first[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int q = 0; q < sep_waves(); q++) s += first[q];
        partial[blockIdx.x + (long)gridDim.x * m] = s;
    }
}

// x(i, j, k) = or += sum_lm V_x[i][l] V_y[j][m] w(l, m, k) for the rows j of a
// block of 16 nb from tile t0 (of the tiles below t1) and plane k = k0 +
// blockIdx.y; columns of the tiles [i0, i1). pinned: plus the constant that
// gives cell (0, 0, 0) its right-hand side (np partial sums of its value).
// flag: solid cells take b.
template <int MR, int NR>
__global__ void __launch_bounds__(kSepThreads) k_sep_back(Dims d, SeparableBatch B, int nb, int t0, int t1, int i0, int i1,
                                                          int k0, int add, int pinned, const double *b,
                                                          const uint8_t *flag, const double *partial, int np) {
    extern __shared__ double sep_lds[];
    __shared__ double first[kSepWaves];
    const SeparableAxis &X = B.S[blockIdx.z].ax[0], &Y = B.S[blockIdx.z].ax[1];
    const double *w_in = B.in[blockIdx.z];
    double *x = B.out[blockIdx.z];
    const int wave = threadIdx.x >> 6, ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = k0 + blockIdx.y, j0 = 16 * (t0 + blockIdx.x * nb), pitch = X.np + kSepPadRow;
    const int xt = X.np / 16, jt = min(nb, t1 - j0 / 16);
    double base = 0;
    if (pinned) {
        double s = 0;
        for (int q = threadIdx.x; q < np; q += blockDim.x) s += partial[q];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if ((threadIdx.x & 63) == 0) first[wave] = s;
    }
    sep_macro<MR, NR>(jt, xt, [&](int jr, int n) {
        const double *vy[MR], *col[NR];
        for (int r = 0; r < MR; r++) vy[r] = Y.V + (long)(j0 + 16 * min(jr + r, jt - 1) + ln) * Y.np + 2 * g;
        for (int s = 0; s < NR; s++) col[s] = w_in + cidx(d, min(16 * (n + s) + ln, d.nx - 1), 0, k);
        mfma_acc t[MR][NR];
        sep_tiles<MR, NR>(
            Y.np / 16, [&](int r, int m, double (&v)[4]) { sep_row(vy[r] + m, v); },
            [&](int s, int m, double (&v)[4]) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = col[s][(long)min(m + sep_k(g, e), d.ny - 1) * d.sy];
            },
            t);
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int s = 0; s < NR; s++)
                if (jr + r < jt && n + s < xt)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        sep_lds[(16 * (jr + r) + 4 * e + g) * pitch + 16 * (n + s) + ln] = t[r][s][e];
    });
    __syncthreads();
    if (pinned) {
        double s = 0;
        for (int q = 0; q < sep_waves(); q++) s += first[q];
        base = b[cidx(d, 0, 0, 0)] - s;
    }
    sep_macro<MR, NR>(jt, i1 - i0, [&](int jr, int n) {
        const double *vx[NR], *row[MR];
        for (int r = 0; r < MR; r++) row[r] = sep_lds + (16 * min(jr + r, jt - 1) + ln) * pitch + 2 * g;
        for (int s = 0; s < NR; s++) vx[s] = X.V + (long)(16 * min(i0 + n + s, i1 - 1) + ln) * X.np + 2 * g;
        mfma_acc t[MR][NR];
        sep_tiles<MR, NR>(
            xt, [&](int r, int l, double (&v)[4]) { sep_row(row[r] + l, v); },
            [&](int s, int l, double (&v)[4]) { sep_row(vx[s] + l, v); }, t);
#pragma unroll
        for (int r = 0; r < MR; r++)
#pragma unroll
            for (int s = 0; s < NR; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int i = 16 * (i0 + n + s) + ln, j = j0 + 16 * (jr + r) + 4 * e + g;
                    if (jr + r >= jt || i0 + n + s >= i1 || i >= d.nx || j >= d.ny) continue;
                    const long q = cidx(d, i, j, k);
                    const double v = flag && flag[q] == F_SOLID ? b[q] : t[r][s][e] + base;
                    x[q] = add ? x[q] + v : v;
                }
    });
}

static int sep_pad16(int n) { return (n + 15) / 16 * 16; }

// LDS tile of a workgroup, at most half a compute unit's: two workgroups share
// one up to a few bytes less (k_sep_z's 64 static bytes leave one at exactly
// half: 256 cells in z). With 64 KB the last kernel takes 103 us at 256 x 128 x
// 128 instead of 71: two row tiles need 66 KB.
constexpr size_t kSepLds = 80 * 1024;

// Row pitch of a column-read tile of nb tiles of 16 beside a padded axis of np
// (less padding on the longest axes), and the LDS of a block in its larger
// layout: np rows of 16 nb, or 16 nb rows of np
static int sep_pitch(int nb, int np) {
    return 16 * nb + (np * (16 * nb + kSepPadCol) * sizeof(double) <= kSepLds ? kSepPadCol : kSepPadCol / 2);
}
static size_t sep_lds_bytes(int nb, int np) {
    return std::max((size_t)np * sep_pitch(nb, np), (size_t)16 * nb * (np + kSepPadRow)) * sizeof(double);
}

// Tiles of 16 per block along an axis of `tiles` tiles beside `other` blocks
// of the grid: as many as leave a workgroup for every compute unit and fit
// the LDS, up to four (the operands are then read by fewer workgroups).
static int sep_block(int tiles, int other, int np) {
    for (int nb = 4; nb > 1; nb /= 2)
        if (tiles >= nb && (long)((tiles + nb - 1) / nb) * other >= 256 && sep_lds_bytes(nb, np) <= kSepLds) return nb;
    return 1;
}

bool separable_fits(const int n[3]) {
    return sep_lds_bytes(1, sep_pad16(std::max({n[0], n[1], n[2]}))) <= kSepLds;
}

long separable_partials(const Dims &d) { return (long)(sep_pad16(d.nx) / 16) * d.ny; }

// Calls f with the macro tile for mt x nt tiles per workgroup and the threads:
// 2 x 2 where that leaves one for each of four waves, else 2 tiles along the
// longer side (rows: the first two kernels, columns: the last), else 1 x 1;
// eight waves where there are macro tiles for them and the grid alone does not
// fill the chip. Last kernel, canopy 160 x 80 x 48: 28 us with 1 x 1 and four
// waves, 19 with 1 x 2 and eight.
template <int N> using SepInt = std::integral_constant<int, N>;
template <typename F>
static void sep_shape(int mt, int nt, bool rows, long groups, F f) {
    const int m2 = (mt + 1) / 2, n2 = (nt + 1) / 2;
    const auto threads = [&](int tiles) { return groups < 1024 && tiles > 4 ? 512 : 256; };
    if (mt > 1 && nt > 1 && m2 * n2 >= 4) f(SepInt<2>(), SepInt<2>(), threads(m2 * n2));
    else if (rows && m2 * nt >= 3) f(SepInt<2>(), SepInt<1>(), threads(m2 * nt));
    else if (!rows && mt * n2 >= 3) f(SepInt<1>(), SepInt<2>(), threads(mt * n2));
    else f(SepInt<1>(), SepInt<1>(), threads(mt * nt));
}

struct SepRange { int i0, i1, j0, j1, k0, k1; };  // cells; i and j in whole tiles of 16

template <int WHAT>
static void sep_xy(hipStream_t st, const Dims &d, int n, const SeparableBatch &B, const uint16_t *mask,
                   const SepRange &in) {
    const int xt = B.S[0].ax[0].np / 16, np = B.S[0].ax[1].np, nk = in.k1 - in.k0;
    const int nb = sep_block(xt, nk * n, np), gx = (xt + nb - 1) / nb, pitch = sep_pitch(nb, np);
    sep_shape(np / 16, nb, true, (long)gx * nk * n, [&](auto mr, auto nr, int threads) {
        hipLaunchKernelGGL((k_sep_xy<WHAT, mr(), nr()>), dim3(gx, nk, n), dim3(threads),
                           (size_t)np * pitch * sizeof(double), st, d, B, mask, nb, pitch, in.k0, in.i0 / 16,
                           (in.i1 + 15) / 16, in.j0 / 16, (in.j1 + 15) / 16);
    });
}

// planes [k0, k1) (whole tiles of 16); returns the number of partial sums
template <bool UNIT>
static int sep_z(hipStream_t st, const Dims &d, int n, const SeparableBatch &B, int k0, int k1, int ku,
                 double *partial) {
    const int xt = B.S[0].ax[0].np / 16, np = B.S[0].ax[2].np;
    const int nb = sep_block(xt, d.ny * n, np), g = (xt + nb - 1) / nb, pitch = sep_pitch(nb, np);
    sep_shape(np / 16, nb, true, (long)g * d.ny * n, [&](auto mr, auto nr, int threads) {
        hipLaunchKernelGGL((k_sep_z<UNIT, mr(), nr()>), dim3(g, d.ny, n), dim3(threads),
                           (size_t)np * pitch * sizeof(double), st, d, B, nb, pitch, k0 / 16, (k1 + 15) / 16, ku,
                           partial);
    });
    return g * d.ny;
}

static void sep_back(hipStream_t st, const Dims &d, int n, const SeparableBatch &B, const SepRange &o, bool add,
                     const double *b, const uint8_t *flag, const double *partial, int partials) {
    const int t0 = o.j0 / 16, t1 = (o.j1 + 15) / 16, nk = o.k1 - o.k0, np = B.S[0].ax[0].np;
    const int nb = sep_block(t1 - t0, nk * n, np), gy = (t1 - t0 + nb - 1) / nb;
    sep_shape(nb, np / 16, false, (long)gy * nk * n, [&](auto mr, auto nr, int threads) {
        hipLaunchKernelGGL((k_sep_back<mr(), nr()>), dim3(gy, nk, n), dim3(threads),
                           (size_t)16 * nb * (np + kSepPadRow) * sizeof(double), st, d, B, nb, t0, t1, o.i0 / 16,
                           (o.i1 + 15) / 16, o.k0, add ? 1 : 0, partial ? B.S[0].pinned : 0, b, flag, partial,
                           partials);
    });
}

void launch_separable_batch(hipStream_t st, const Dims &d, int n, const SeparableSys *S, const double *const *b,
                            double *const *s1, double *const *s2, double *const *x) {
    SeparableBatch B[3]{};
    for (int c = 0; c < n; c++)
        for (int p = 0; p < 3; p++) {
            B[p].S[c] = S[c];
            B[p].in[c] = p == 0 ? b[c] : p == 1 ? s1[c] : s2[c];
            B[p].out[c] = p == 0 ? s1[c] : p == 1 ? s2[c] : x[c];
        }
    const SepRange all{0, d.nx, 0, d.ny, 0, d.nz};
    sep_xy<SEP_ALL>(st, d, n, B[0], nullptr, all);
    sep_z<false>(st, d, n, B[1], 0, d.nz, 0, nullptr);
    sep_back(st, d, n, B[2], all, false, nullptr, nullptr, nullptr, 0);
}

void launch_separable(hipStream_t st, const Dims &d, const SeparableSys &S, const double *b, double *s1, double *s2,
                      double *x, bool add, double *partial) {
    const SepRange all{0, d.nx, 0, d.ny, 0, d.nz};
    sep_xy<SEP_ALL>(st, d, 1, {{S}, {b}, {s1}}, nullptr, all);
    const int np = sep_z<false>(st, d, 1, {{S}, {s1}, {s2}}, 0, d.nz, 0, partial);
    sep_back(st, d, 1, {{S}, {s2}, {x}}, all, add, b, nullptr, partial, np);
}

// ---------------------------------------------------------------------------
// immersed body
// ---------------------------------------------------------------------------
// One solve is two passes of the transforms, the first one's last two limited
// to the planes and rows the ghost rows look at, and one product with the
// inverse of the ghost rows' matrix: 256 x 128 x 128 with 3568 ghost cells
// 0.34 ms, of it 32 us for the product (102 MB); BiCGSTAB with multigrid
// cycles took 7 iterations of 0.95 ms.
// Row s of R at y, a: its sum over the stencil points. Where a cell centre lies
// on the surface the mirror point is the cell itself and the row is zero (up to
// rounding of its weights): p' keeps its start value there, so the row is x = b.
__device__ inline double cap_row(const GhostRows<double> &G, int s, double yc, double a) {
    const double dg = 1 - G.wself[s];
    return dg != 0 ? dg * yc - a : yc;
}

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
    t[s] = b[c] - cap_row(G, s, y[c], a);
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
    const SepRange all{0, d.nx, 0, d.ny, 0, d.nz};
    const SepRange look{B.look.lo[0], B.look.hi[0], B.look.lo[1], B.look.hi[1], B.look.lo[2], B.look.hi[2]};
    const SepRange cells{B.cells.lo[0], B.cells.hi[0], B.cells.lo[1], B.cells.hi[1], B.cells.lo[2], B.cells.hi[2]};
    sep_xy<SEP_MASK>(st, d, 1, {{S}, {b}, {s1}}, B.fluid, all);
    sep_z<false>(st, d, 1, {{S}, {s1}, {s2}}, look.k0, look.k1, 0, nullptr);
    sep_back(st, d, 1, {{S}, {s2}, {s3}}, look, false, b, nullptr, nullptr, 0);
    const int ng = B.G.ng;
    hipLaunchKernelGGL(k_cap_rhs, dim3((ng + 63) / 64), dim3(64), 0, st, B.G, b, s3, B.t);
    if (B.inv64)
        hipLaunchKernelGGL((k_cap_apply<double>), dim3((ng + 3) / 4), dim3(256), 0, st, B.G, B.inv64, B.ld, B.t, s3);
    else
        hipLaunchKernelGGL((k_cap_apply<float>), dim3((ng + 3) / 4), dim3(256), 0, st, B.G, B.inv32, B.ld, B.t, s3);
    sep_xy<SEP_ADD>(st, d, 1, {{S}, {s3}, {s1}}, B.ghost, cells);
    sep_z<false>(st, d, 1, {{S}, {s1}, {s2}}, 0, d.nz, 0, nullptr);
    sep_back(st, d, 1, {{S}, {s2}, {x}}, all, add, b, B.flag, nullptr, 0);
}

// A^-1 e_c in the box, for the unit vectors of the ghost cells c = src0 +
// blockIdx.z of one plane: h holds their common z part (k_sep_z<true>), the
// x and y parts scale the last two transforms' matrices. Rows: 16 from y tile
// box.lo[1] / 16 + blockIdx.x, plane box.lo[2] + blockIdx.y.
__global__ void __launch_bounds__(kSepThreads) k_cap_green(Dims d, SeparableAxis X, SeparableAxis Y, const double *h,
                                                           const int3 *src, int src0, GreenBox box,
                                                           GreenScratch out) {
    extern __shared__ double sep_lds[];
    const int ln = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int k = box.lo[2] + blockIdx.y, j0 = 16 * (box.lo[1] / 16 + blockIdx.x), pitch = X.np + kSepPadRow;
    const int xt = X.np / 16, x0 = box.lo[0] / 16, x1 = (box.hi[0] + 15) / 16;
    const int3 c = src[src0 + blockIdx.z];
    double *fy = sep_lds + 16 * pitch;  // Vi_y[m][j of the source]
    for (int m = threadIdx.x; m < Y.np; m += blockDim.x) fy[m] = Y.Vi[(long)m * Y.np + c.y];
    __syncthreads();
    sep_macro<1, 2>(1, xt, [&](int, int n) {
        const double *vy = Y.V + (long)(j0 + ln) * Y.np + 2 * g, *col[2];
        for (int s = 0; s < 2; s++) col[s] = h + cidx(d, min(16 * (n + s) + ln, d.nx - 1), 0, k);
        mfma_acc t[1][2];
        sep_tiles<1, 2>(
            Y.np / 16, [&](int, int m, double (&v)[4]) { sep_row(vy + m, v); },
            [&](int s, int m, double (&v)[4]) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int q = m + sep_k(g, e);
                    v[e] = col[s][(long)min(q, d.ny - 1) * d.sy] * fy[q];
                }
            },
            t);
        for (int s = 0; s < 2 && n + s < xt; s++) {
            const int l = 16 * (n + s) + ln;
            const double fx = X.Vi[(long)l * X.np + c.x];
#pragma unroll
            for (int e = 0; e < 4; e++) sep_lds[(4 * e + g) * pitch + l] = t[0][s][e] * fx;
        }
    });
    __syncthreads();
    const int bx = box.hi[0] - box.lo[0], by = box.hi[1] - box.lo[1], bz = box.hi[2] - box.lo[2];
    double *o = out.v[blockIdx.z / out.per] + (long)(blockIdx.z % out.per) * bx * by * bz
        + (long)(k - box.lo[2]) * bx * by;
    sep_macro<1, 1>(1, x1 - x0, [&](int, int n) {
        const int i = 16 * (x0 + n) + ln;
        const double *vx = X.V + (long)i * X.np + 2 * g, *row = sep_lds + ln * pitch + 2 * g;
        mfma_acc t[1][1];
        sep_tiles<1, 1>(
            xt, [&](int, int l, double (&v)[4]) { sep_row(row + l, v); },
            [&](int, int l, double (&v)[4]) { sep_row(vx + l, v); }, t);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int j = j0 + 4 * e + g;
            if (i >= box.lo[0] && i < box.hi[0] && j >= box.lo[1] && j < box.hi[1])
                o[(long)(j - box.lo[1]) * bx + i - box.lo[0]] = t[0][0][e];
        }
    });
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
    out[s * ld + src[src0 + c].z] = cap_row(G, s, y[loc[9 * (long)s + 8]], a);
}

void launch_green_plane(hipStream_t st, const Dims &d, const SeparableSys &S, int k, const int3 *src, int nsrc,
                        const GreenBox &box, const GhostRows<double> &G, const int *loc, double *h,
                        const GreenScratch &green, double *out, long ld) {
    const long vol = (long)(box.hi[0] - box.lo[0]) * (box.hi[1] - box.lo[1]) * (box.hi[2] - box.lo[2]);
    sep_z<true>(st, d, 1, {{S}, {h}, {h}}, box.lo[2], box.hi[2], k, nullptr);
    const int jt = (box.hi[1] + 15) / 16 - box.lo[1] / 16, batch = kGreenVecs * green.per;
    for (int c = 0; c < nsrc; c += batch) {
        const int n = std::min(batch, nsrc - c);
        hipLaunchKernelGGL(k_cap_green, dim3(jt, box.hi[2] - box.lo[2], n), dim3(256),
                           (16 * (size_t)(S.ax[0].np + kSepPadRow) + S.ax[1].np) * sizeof(double), st, d, S.ax[0],
                           S.ax[1], h, src, c, box, green);
        hipLaunchKernelGGL(k_cap_rows, dim3((G.ng + 255) / 256, n), dim3(256), 0, st, G, loc, src, c, vol, green, out,
                           ld);
    }
}

// *bad = 1 where a value is not finite: reads the inverse once (n = 6579, 346 MB:
// 0.1 ms)
template <typename T>
__global__ void __launch_bounds__(256) k_not_finite(const T *a, long n, int *bad) {
    bool any = false;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += 256L * gridDim.x) any |= !isfinite(a[e]);
    if (any) *bad = 1;
}

template <typename T>
void launch_not_finite(hipStream_t st, const T *a, long n, int *bad) {
    hipLaunchKernelGGL((k_not_finite<T>), dim3((unsigned)std::min(4096L, (n + 255) / 256)), dim3(256), 0, st, a, n,
                       bad);
}
template void launch_not_finite<float>(hipStream_t, const float *, long, int *);
template void launch_not_finite<double>(hipStream_t, const double *, long, int *);

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

bool separable_axis(int n, bool periodic, const std::vector<double> coef[4], std::vector<double> &V,
                    std::vector<double> &Vi, std::vector<double> &lam) {
    const std::vector<double> &cm = coef[0], &cp = coef[1], &dm = coef[2], &dp = coef[3];
    std::vector<double> q, ev, w(n, 1.0);  // w: square roots of the weights
    if (periodic) {
        // uniform spacing: Fourier modes
        for (int i = 0; i < n; i++)
            if (std::fabs(cm[i] - cm[0]) > 1e-10 * cm[0] || std::fabs(cp[i] - cm[0]) > 1e-10 * cm[0]) return false;
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
            // weight_i cp_i = weight_(i+1) cm_(i+1): the operator is symmetric
            if (!(cp[i] > 0) || !(cm[i + 1] > 0)) return false;
            w[i + 1] = w[i] * std::sqrt(cp[i] / cm[i + 1]);
            e[i] = -std::sqrt(cp[i] * cm[i + 1]);
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
            V[(size_t)i * np + m] = z / w[i];
            Vi[(size_t)m * np + i] = z * w[i];
        }
    }
    return true;
}

}  // namespace ibm
