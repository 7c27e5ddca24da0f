// step_kernels.hip - stencil kernels of one fractional step (FP64).
//
// Each kernel restates one stage of the reference's IBMSolver_iterate
// (src/ibm3d_fracstep.c) for the x-contiguous device layout of common.h:
//   k_interp_stag    interp_stag_vel            :807-845
//   k_conv_rhs       calc_N + momentum RHS      :117-170, :225-269
//   k_face_star      calc_u_tilde + calc_U_star :388-487 (u~ formed on the fly)
//   k_poisson_rhs    pressure RHS               :539-552
//   k_update         update_next                :709-792
//   k_outer_*        update_outer               :855-1906
//   k_ghost_*        update_ghost               :1915-1976
//   k_sgs            Smagorinsky / Vreman stress src/ibm3d_turb.c:8-82
// One thread per cell; blocks of 64 (x) by 4 (y) threads so a wavefront reads
// one 512-byte x-row segment per array.
#include "step_kernels.h"

#include <algorithm>

namespace ibm {

#define C1(a, i) ((a)[(i) + 2])

// v is formed here, by every lane: else the compiler turns a select of it into a
// branch, its loads behind that, one round trip to memory after another
__device__ inline void form_now(double &v) { asm volatile("" : "+v"(v)); }

__device__ inline double nan_d() { return __builtin_nan(""); }

// ---------------------------------------------------------------------------
// block reduction of NV doubles into partial[blockLinear * NV + v]
// ---------------------------------------------------------------------------
template <int NV>
__device__ inline void block_sum_store(double (&v)[NV], double *partial, long blk) {
    __shared__ double sh[NV][16];
    const int tid = threadIdx.x + threadIdx.y * blockDim.x + threadIdx.z * blockDim.x * blockDim.y;
    const int nth = blockDim.x * blockDim.y * blockDim.z;
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int a = 0; a < NV; a++) {
        double x = v[a];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o, 64);
        if (lane == 0) sh[a][wave] = x;
    }
    __syncthreads();
    if (tid == 0) {
        const int nw = (nth + 63) >> 6;
#pragma unroll
        for (int a = 0; a < NV; a++) {
            double acc = 0;
            for (int w = 0; w < nw; w++) acc += sh[a][w];
            partial[blk * NV + a] = acc;
        }
    }
}

__device__ inline long block_linear() {
    return blockIdx.x + (long)gridDim.x * (blockIdx.y + (long)gridDim.y * blockIdx.z);
}

// ---------------------------------------------------------------------------
// interp_stag_vel: face velocities from cell velocities over the padded
// tangential extent.  <- src/ibm3d_fracstep.c:807-845
// ---------------------------------------------------------------------------
__global__ void k_interp_stag(Geo g, const double *u1, const double *u2, const double *u3,
                              double *U1, double *U2, double *U3) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x - 2;
    const int j = blockIdx.y * blockDim.y + threadIdx.y - 2;
    const int k = blockIdx.z - 2;
    if (i > d.nx + 1 || j > d.ny + 1) return;
    const long q = cidx(d, i, j, k);
    if (i >= 0 && i <= d.nx)
        U1[q] = (u1[q - 1] * C1(g.dx, i) + u1[q] * C1(g.dx, i - 1)) / (C1(g.dx, i - 1) + C1(g.dx, i));
    if (j >= 0 && j <= d.ny)
        U2[q] = (u2[q - d.sy] * C1(g.dy, j) + u2[q] * C1(g.dy, j - 1)) / (C1(g.dy, j - 1) + C1(g.dy, j));
    if (k >= 0 && k <= d.nz)
        U3[q] = (u3[q - d.sz] * C1(g.dz, k) + u3[q] * C1(g.dz, k - 1)) / (C1(g.dz, k - 1) + C1(g.dz, k));
}

// ---------------------------------------------------------------------------
// K1: convection N (AB2 history) and the Crank-Nicolson momentum RHS of the
// three components, fused.  <- src/ibm3d_fracstep.c:117-170 and :237-269
// Writes N (non-fluid: NaN) and b_l (non-fluid rows: 0); accumulates the
// squared norms of b_l over the interior rows for the stopping test. Bound by
// its 16 fields: 256 x 128 x 128 166 us, 3.3 TB/s of those, 4.2 with the halos
// (175 with the components one after the other: a store between them, or a
// branch on the turbulence stress or the forcing, holds the next one's loads
// back, hence the two switches at compile time and the stores at the end; 187
// with the 30 divisions per cell that the axis metrics replace; the blocks in
// contiguous ranges per XCD: 8 us more; several planes per thread, 212 registers).
// ---------------------------------------------------------------------------
template <bool TAU, bool FA>
__global__ void __launch_bounds__(256) k_conv_rhs(Geo g, StepParams sp, const uint8_t *flag,
                                                  const double *u1, const double *u2, const double *u3,
                                                  const double *U1, const double *U2, const double *U3,
                                                  const double *p, const double *Np1, const double *Np2,
                                                  const double *Np3, double *N1, double *N2, double *N3,
                                                  double *b1, double *b2, double *b3, TauPtrs tau,
                                                  double *partial) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    double nrm[3] = {0, 0, 0};
    if (i < d.nx && j < d.ny) {
        // every cell is computed (the neighbours of interior cells are in the
        // padded range) and non-fluid results are replaced at the end, so all
        // loads issue before the first wait
        const long q = cidx(d, i, j, k);
        const long sy = d.sy, sz = d.sz;
        const bool fl = flag[q] == F_FLUID;
        const AxisMetric X0 = C1(g.mx, i), Y0 = C1(g.my, j), Z0 = C1(g.mz, k);
        const double wxp = C1(g.mx, i + 1).w, wyp = C1(g.my, j + 1).w, wzp = C1(g.mz, k + 1).w;
        const double Uw = U1[q], Ue = U1[q + 1], Vs = U2[q], Vn = U2[q + sy], Wd = U3[q], Wu = U3[q + sz];
        const double kW = C1(g.kW, i), kE = C1(g.kE, i), kS = C1(g.kS, j), kN = C1(g.kN, j);
        const double kD = C1(g.kD, k), kU = C1(g.kU, k);
        const double kc = 1 - kW - kE - kS - kN - kD - kU;
        const double *uu[3] = {u1, u2, u3};
        const double *Np[3] = {Np1, Np2, Np3};
        double *NN[3] = {N1, N2, N3};
        double *bb[3] = {b1, b2, b3};
        const double dp[3] = {(p[q + 1] - p[q - 1]) * X0.r2, (p[q + sy] - p[q - sy]) * Y0.r2,
                              (p[q + sz] - p[q - sz]) * Z0.r2};
        double nv[3], bv[3];
#pragma unroll
        for (int l = 0; l < 3; l++) {
            const double *a = uu[l];
            const double c = a[q], xm = a[q - 1], xp = a[q + 1], ym = a[q - sy], yp = a[q + sy];
            const double zm = a[q - sz], zp = a[q + sz];
            const double npl = Np[l][q];
            const double uw = c + X0.w * (xm - c), ue = xp + wxp * (c - xp);
            const double us = c + Y0.w * (ym - c), un = yp + wyp * (c - yp);
            const double ud = c + Z0.w * (zm - c), uu_ = zp + wzp * (c - zp);
            double n = (Ue * ue - Uw * uw) * X0.rd + (Vn * un - Vs * us) * Y0.rd + (Wu * uu_ - Wd * ud) * Z0.rd;
            double divt = 0;
            if (TAU) {
                const double *t1 = tau.t[tau.slot[l][0]], *t2 = tau.t[tau.slot[l][1]], *t3 = tau.t[tau.slot[l][2]];
                divt = (t1[q + 1] - t1[q - 1]) * X0.r2 + (t2[q + sy] - t2[q - sy]) * Y0.r2
                    + (t3[q + sz] - t3[q - sz]) * Z0.r2;
            }
            double b = -sp.dt / 2 * (3 * n - npl) - sp.dt * dp[l] + kc * c
                + kW * xm + kE * xp + kS * ym + kN * yp + kD * zm + kU * zp
                + sp.dt * (FA && sp.fa[l] ? sp.fa[l][q] : sp.force[l]) - sp.dt * divt;
            form_now(n);
            form_now(b);
            nv[l] = fl ? n : nan_d();
            bv[l] = fl ? b : 0.0;
        }
#pragma unroll
        for (int l = 0; l < 3; l++) {
            NN[l][q] = nv[l];
            bb[l][q] = bv[l];
            nrm[l] = bv[l] * bv[l];
        }
    }
    block_sum_store<3>(nrm, partial, block_linear());
}

// ---------------------------------------------------------------------------
// K2a: predicted face velocities U*.  <- src/ibm3d_fracstep.c:388-487
// U* = interp(u~) - dt dp/dn with u~ = u* + dt grad p (central), except on
// fluid|ghost faces where U* = interp(u*). Threads cover (nx+1)(ny+1)(nz+1)
// cells; cell (i,j,k) owns its three low faces.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_face_star(Geo g, StepParams sp, const uint8_t *flag,
                                                   const double *us1, const double *us2, const double *us3,
                                                   const double *p, double *F1, double *F2, double *F3) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i > d.nx || j > d.ny) return;
    const long q = cidx(d, i, j, k);
    const long sy = d.sy, sz = d.sz;
    const double dt = sp.dt;
    // every load is in the padded range: all issue before the first wait, and
    // the faces past the last cell's are dropped at the stores
    const uint8_t f0 = flag[q], fx = flag[q - 1], fy = flag[q - sy], fz = flag[q - sz];
    const double p0 = p[q];
    const double px[3] = {p[q - 2], p[q - 1], p[q + 1]}, py[3] = {p[q - 2 * sy], p[q - sy], p[q + sy]};
    const double pz[3] = {p[q - 2 * sz], p[q - sz], p[q + sz]};
    const double ux = us1[q - 1], vx = us1[q], uy = us2[q - sy], vy = us2[q], uz = us3[q - sz], vz = us3[q];
    const AxisMetric X = C1(g.mx, i), Y = C1(g.my, j), Z = C1(g.mz, k);
    const double xr = C1(g.mx, i - 1).r2, yr = C1(g.my, j - 1).r2, zr = C1(g.mz, k - 1).r2;
    const auto face = [&](uint8_t fm, const AxisMetric &M, double rm, double um, double u0, const double (&pn)[3]) {
        const double tm = um + dt * (p0 - pn[0]) * rm, t0 = u0 + dt * (pn[2] - pn[1]) * M.r2;
        const bool body = fm + f0 == F_FLUID + F_GHOST && fm != f0;
        double vb = u0 + M.w * (um - u0), v = t0 + M.w * (tm - t0) - dt * (p0 - pn[1]) * M.rc;
        form_now(vb);
        form_now(v);
        return body ? vb : v;
    };
    const double v1 = face(fx, X, xr, ux, vx, px), v2 = face(fy, Y, yr, uy, vy, py), v3 = face(fz, Z, zr, uz, vz, pz);
    if (j < d.ny && k < d.nz) F1[q] = v1;
    if (i < d.nx && k < d.nz) F2[q] = v2;
    if (i < d.nx && j < d.ny) F3[q] = v3;
}

// ---------------------------------------------------------------------------
// K2b: pressure-correction RHS b = -(1/2Re) div U* on fluid rows (the
// reference divides it by the diagonal sum K, :545-550; the solver here keeps
// the unnormalised row and applies that scaling only in the stopping test).
// Accumulates ||b / sum K||^2.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_poisson_rhs(Geo g, StepParams sp, const uint8_t *flag, long pin,
                                                     const double *F1, const double *F2, const double *F3,
                                                     double *b, double *partial) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    double nrm[1] = {0};
    if (i < d.nx && j < d.ny) {
        const long q = cidx(d, i, j, k);
        double v = 0;
        if (q != pin && flag[q] == F_FLUID) {
            v = -1 / (2 * sp.Re) * ((F1[q + 1] - F1[q]) * C1(g.mx, i).rd + (F2[q + d.sy] - F2[q]) * C1(g.my, j).rd
                                    + (F3[q + d.sz] - F3[q]) * C1(g.mz, k).rd);
            const double ks = C1(g.kN, j) + C1(g.kE, i) + C1(g.kS, j) + C1(g.kW, i) + C1(g.kD, k) + C1(g.kU, k);
            const double vn = v / ks;
            nrm[0] = vn * vn;
        }
        b[q] = v;
    }
    block_sum_store<1>(nrm, partial, block_linear());
}

// ---------------------------------------------------------------------------
// K3: projection.  <- src/ibm3d_fracstep.c:740-792
// p_next = p + p' (fluid, ghost) / NaN (solid); u_next = u* - dt grad p'
// (fluid) / NaN (solid); ghost entries of u_next are left untouched, as in
// the reference. U_next = U* - dt dp'/dn on faces with no solid side, else NaN.
// 256 x 128 x 128: 106 us, 6.1 TB/s (121 with the flags looked at before each
// load).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_update(Geo g, StepParams sp, const uint8_t *flag,
                                                const double *p, const double *pp,
                                                const double *us1, const double *us2, const double *us3,
                                                const double *F1, const double *F2, const double *F3,
                                                double *pn, double *un1, double *un2, double *un3,
                                                double *G1, double *G2, double *G3) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i > d.nx || j > d.ny) return;
    const long q = cidx(d, i, j, k);
    const long sy = d.sy, sz = d.sz;
    const double dt = sp.dt;
    // every load is in the padded range: all issue before the first wait
    const uint8_t f0 = flag[q], fx = flag[q - 1], fy = flag[q - sy], fz = flag[q - sz];
    const double pc = p[q], c = pp[q], xm = pp[q - 1], xp = pp[q + 1], ym = pp[q - sy], yp = pp[q + sy];
    const double zm = pp[q - sz], zp = pp[q + sz];
    const double u1 = us1[q], u2 = us2[q], u3 = us3[q], s1 = F1[q], s2 = F2[q], s3 = F3[q];
    const AxisMetric X = C1(g.mx, i), Y = C1(g.my, j), Z = C1(g.mz, k);
    const bool in0 = f0 != F_SOLID;
    double pv = pc + c, n1 = u1 - dt * (xp - xm) * X.r2, n2 = u2 - dt * (yp - ym) * Y.r2;
    double n3 = u3 - dt * (zp - zm) * Z.r2;
    double g1 = s1 - dt * (c - xm) * X.rc, g2 = s2 - dt * (c - ym) * Y.rc, g3 = s3 - dt * (c - zm) * Z.rc;
    for (double *v : {&pv, &n1, &n2, &n3, &g1, &g2, &g3}) form_now(*v);
    const bool fluid = f0 == F_FLUID;
    pv = fluid || f0 == F_GHOST ? pv : nan_d();
    n1 = fluid ? n1 : nan_d();
    n2 = fluid ? n2 : nan_d();
    n3 = fluid ? n3 : nan_d();
    g1 = in0 && fx != F_SOLID ? g1 : nan_d();
    g2 = in0 && fy != F_SOLID ? g2 : nan_d();
    g3 = in0 && fz != F_SOLID ? g3 : nan_d();
    if (i < d.nx && j < d.ny && k < d.nz) {
        pn[q] = pv;
        if (fluid || f0 == F_SOLID) {
            un1[q] = n1;
            un2[q] = n2;
            un3[q] = n3;
        }
    }
    if (j < d.ny && k < d.nz) G1[q] = g1;
    if (i < d.nx && k < d.nz) G2[q] = g2;
    if (i < d.nx && j < d.ny) G3[q] = g3;
}

// ---------------------------------------------------------------------------
// Outer boundary layers.  <- src/ibm3d_fracstep.c:855-1906
// One launch for the six faces and all fields. The reference fills x, then y,
// then z faces, each reading the corner values that the previous ones wrote;
// here a thread evaluates those itself: an outer value is a constant plus at
// most two values further in on its axis, which may in turn be outer on an
// earlier axis. Tangential ranges as in the reference: x faces (j, k)
// interior; y faces i padded, k interior; z faces i, j padded. One value per
// thread, its rule read from a table made at assembly: bound by the launch and
// a chain of dependent loads. 32^3: 5.8 us for the four fields, 3 launches per
// step (a launch per axis was 12 of 5.6 us); rules evaluated in the kernel, all
// layers and fields in one thread, took 33 us.
// ---------------------------------------------------------------------------
__device__ inline double bcval(const FaceBC &f, int comp, int t1, int t2, int n2) {
    if (f.garr) return f.garr[((long)comp * f.n1 + (t1 + f.t1off)) * n2 + (t2 + f.t2off)];
    return f.g[comp];
}

// value of f at (i, j, k), outer positions on the axes up to AX evaluated;
// rules: of f's kind
template <int AX>
__device__ inline double outer_value(const Dims &d, const OuterParams &op, const OuterRule *rules, const double *f,
                                     int comp, int i, int j, int k) {
    const int n = AX == 0 ? i : AX == 1 ? j : k, N = AX == 0 ? d.nx : AX == 1 ? d.ny : d.nz;
    if (n >= 0 && n < N) {
        if constexpr (AX == 0) return f[cidx(d, i, j, k)];
        else return outer_value<AX - 1>(d, op, rules, f, comp, i, j, k);
    }
    const int hi = n >= N, layer = hi ? n - N : -1 - n;
    const OuterRule &r = rules[(2 * AX + hi) * 2 + layer];
    if (r.keep) return f[cidx(d, i, j, k)];
    double v = 0;
    if (r.g != 0)
        v = r.g * bcval(op.face[AX][hi], comp, AX == 0 ? j : i, AX == 2 ? j : k, AX == 2 ? d.ny + 4 : d.nz);
#pragma unroll 1
    for (int t = 0; t < 2; t++) {
        const double c = r.c[t];
        if (c == 0) continue;
        const int m = r.n[t], x = AX == 0 ? m : i, y = AX == 1 ? m : j, z = AX == 2 ? m : k;
        // a position that is not interior on this axis (a single cell wide) is taken as it is
        double w;
        if (AX == 0 || m < 0 || m >= N) w = f[cidx(d, x, y, z)];
        else w = outer_value<AX == 0 ? 0 : AX - 1>(d, op, rules, f, comp, x, y, z);
        v += c * w;
    }
    return v;
}

// One workgroup of 256 threads: fixed-order sums. Riding beside a boundary
// launch it costs no launch of its own (5 us on small grids, four per step), and
// there is no chain between the two. The launch lasts as long as its longest
// rider, which is a chain of round trips to memory: the columns are summed in one
// pass. With an outflow face its norms and the right-hand sides' ride together:
// at 256 x 128 x 128 the launch takes 15 us more in place of three launches of 12,
// 6 and 4 us and their gaps (22.0 -> 21.6 ms for ten steps and their read-back).
constexpr int kRiderThreads = 256;
template <int NV>
__device__ inline void run_rider(const double *partial, long nblk, double *out, int t, double *sh) {
    double acc[NV][4];
#pragma unroll
    for (int a = 0; a < NV; a++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[a][u] = 0;
    long b = t;
    for (; b + 3 * kRiderThreads < nblk; b += 4 * kRiderThreads)
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int a = 0; a < NV; a++) acc[a][u] += partial[(b + u * kRiderThreads) * NV + a];
    for (; b < nblk; b += kRiderThreads)
#pragma unroll
        for (int a = 0; a < NV; a++) acc[a][0] += partial[b * NV + a];
#pragma unroll
    for (int a = 0; a < NV; a++) {
        double v = (acc[a][0] + acc[a][1]) + (acc[a][2] + acc[a][3]);
        for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
        if ((t & 63) == 0) sh[t >> 6] = v;
        __syncthreads();
        if (t == 0) out[a] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
        __syncthreads();
    }
}
__device__ inline void run_riders(const SumRiders &sums) {
    __shared__ double sh[kRiderThreads / 64];
    const int t = threadIdx.x + blockDim.x * threadIdx.y;
    for (int e = 0; e < sums.n; e++) {
        const auto &R = sums.r[e];
        if (R.nv == 3) run_rider<3>(R.partial, R.nblk, R.out, t, sh);
        else if (R.nv == 2) run_rider<2>(R.partial, R.nblk, R.out, t, sh);
        else run_rider<1>(R.partial, R.nblk, R.out, t, sh);
    }
    if (t != 0) return;
    __threadfence_system();
    *reinterpret_cast<volatile unsigned *>(sums.epoch_out) = sums.epoch;
}

__device__ inline void save_ghosts(const GhostSave &g, const OuterFields &fs);

__global__ void __launch_bounds__(kRiderThreads) k_outer(Dims d, OuterParams op, const OuterRule *rules,
                                                         OuterFields fs, SumRiders sums, GhostSave save) {
    if ((int)blockIdx.z == 12 * fs.n) {
        if (sums.n > 0 && blockIdx.x == 0 && blockIdx.y == 0) run_riders(sums);
        if (save.ng > 0) save_ghosts(save, fs);
        return;
    }
    // one value per thread: face, layer and field
    const int ax = blockIdx.z % 6 / 2, hi = blockIdx.z % 2, layer = blockIdx.z / 6 % 2, e = blockIdx.z / 12;
    const int a0 = ax == 0 ? 0 : -2, a1 = ax == 0 ? d.ny : d.nx + 2;
    const int b0 = ax == 2 ? -2 : 0, b1 = ax == 2 ? d.ny + 2 : d.nz;
    const int t1 = a0 + blockIdx.x * blockDim.x + threadIdx.x;
    const int t2 = b0 + blockIdx.y * blockDim.y + threadIdx.y;
    if (t1 >= a1 || t2 >= b1) return;
    const int N = ax == 0 ? d.nx : ax == 1 ? d.ny : d.nz;
    const int kind = fs.kind[e], n = hi ? N + layer : -1 - layer;
    double *f = fs.f[e];
    const int i = ax == 0 ? n : t1, j = ax == 0 ? t1 : ax == 1 ? n : t2, k = ax == 2 ? n : t2;
    // (itself where the rule keeps it)
    f[cidx(d, i, j, k)] = outer_value<2>(d, op, rules + 12 * kind, f, min(kind, 3), i, j, k);
}

// ---------------------------------------------------------------------------
// Convective outflow (extension; no counterpart in the reference). The
// face's convection speed comes from one workgroup (fixed-order sums); the
// update of the face values runs one thread per face entry over many
// workgroups, each leaving fixed-order partial sums of its BC-row norms.
// ---------------------------------------------------------------------------
static constexpr int kConvThreads = 1024;

// fixed-order tree sum over the workgroup; every thread gets the result
__device__ inline double conv_block_sum(double v, double *red) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int w = kConvThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

struct ConvFace {
    int a0, a1, b0, b1, n2, q0;
    long ext, st;
    double bi;
};

__device__ inline ConvFace conv_face(const Geo &g, int ax, int hi) {
    const Dims &d = g.d;
    ConvFace f;
    if (ax == 0) { f.a0 = 0; f.a1 = d.ny; f.b0 = 0; f.b1 = d.nz; }
    else if (ax == 1) { f.a0 = -2; f.a1 = d.nx + 2; f.b0 = 0; f.b1 = d.nz; }
    else { f.a0 = -2; f.a1 = d.nx + 2; f.b0 = -2; f.b1 = d.ny + 2; }
    f.n2 = f.b1 - f.b0;
    f.ext = (long)(f.a1 - f.a0) * f.n2;
    const int N = ax == 0 ? d.nx : ax == 1 ? d.ny : d.nz;
    f.q0 = hi ? N - 1 : 0;
    f.st = ax == 0 ? 1 : ax == 1 ? d.sy : d.sz;
    f.bi = C1(ax == 0 ? g.dx : ax == 1 ? g.dy : g.dz, f.q0) / 2;
    return f;
}

// uc_out = the set speed uc, or for uc <= 0 the area-weighted mean outward
// normal component of the face values over the face's interior cells,
// clamped at 0
__global__ void __launch_bounds__(kConvThreads)
k_conv_speed(Geo g, int ax, int hi, double uc, const double *garr, double *uc_out) {
    __shared__ double red[kConvThreads];
    const Dims &d = g.d;
    if (uc <= 0) {
        const ConvFace f = conv_face(g, ax, hi);
        const int m1 = ax == 0 ? d.ny : d.nx, m2 = ax == 2 ? d.ny : d.nz;
        const double *w1 = ax == 0 ? g.dy : g.dx, *w2 = ax == 2 ? g.dy : g.dz;
        double num = 0, den = 0;
        for (long e = threadIdx.x; e < (long)m1 * m2; e += kConvThreads) {
            // (a face has fewer than 2^32 entries)
            const int t1 = (int)((unsigned)e / (unsigned)m2), t2 = (int)((unsigned)e % (unsigned)m2);
            const double A = C1(w1, t1) * C1(w2, t2);
            num += garr[ax * f.ext + (long)(t1 - f.a0) * f.n2 + (t2 - f.b0)] * A;
            den += A;
        }
        num = conv_block_sum(num, red);
        den = conv_block_sum(den, red);
        uc = fmax((hi ? num : -num) / den, 0.0);
    }
    if (threadIdx.x == 0) *uc_out = uc;
}

// init: g = the first interior cell's velocity; otherwise one explicit
// upwind step g <- g - dt uc (g - u_q0) / (d_q0 / 2). One thread per face
// entry; partial[blk * 3 + c] = the block's sum of 2 g_c^2.
__global__ void __launch_bounds__(256)
k_conv_update(Geo g, int ax, int hi, const double *uc_in, double dt, int init, const double *u1, const double *u2,
              const double *u3, double *garr, double *partial) {
    const Dims &d = g.d;
    const ConvFace f = conv_face(g, ax, hi);
    const long e = blockIdx.x * 256L + threadIdx.x;
    double nrm[3] = {0, 0, 0};
    if (e < f.ext) {
        const double uc = init ? 0.0 : *uc_in;
        const int t1 = f.a0 + (int)((unsigned)e / (unsigned)f.n2), t2 = f.b0 + (int)((unsigned)e % (unsigned)f.n2);
        long base;
        if (ax == 0) base = cidx(d, 0, t1, t2);
        else if (ax == 1) base = cidx(d, t1, 0, t2);
        else base = cidx(d, t1, t2, 0);
        const long cq = base + f.q0 * f.st;
        const double *u[3] = {u1, u2, u3};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double uq = u[c][cq];
            double gv = garr[c * f.ext + e];
            gv = init ? uq : gv - dt * uc * (gv - uq) / f.bi;
            garr[c * f.ext + e] = gv;
            nrm[c] = 2 * gv * gv;
        }
    }
    block_sum_store<3>(nrm, partial, blockIdx.x);
}

long conv_outflow_blocks(const Dims &d, int ax) {
    const long ext = ax == 0 ? (long)d.ny * d.nz : ax == 1 ? (long)(d.nx + 4) * d.nz : (long)(d.nx + 4) * (d.ny + 4);
    return (ext + 255) / 256;
}

long launch_conv_outflow(hipStream_t st, const Geo &g, int ax, int hi, double uc, double dt, int init,
                         const double *u1, const double *u2, const double *u3, double *garr, double *uc_slot,
                         double *partial) {
    if (!init) hipLaunchKernelGGL(k_conv_speed, dim3(1), dim3(kConvThreads), 0, st, g, ax, hi, uc, garr, uc_slot);
    const long nblk = conv_outflow_blocks(g.d, ax);
    hipLaunchKernelGGL(k_conv_update, dim3(nblk), dim3(256), 0, st, g, ax, hi, uc_slot, dt, init, u1, u2, u3, garr,
                       partial);
    return nblk;
}

// ---------------------------------------------------------------------------
// Inhomogeneous boundary data folded into the right-hand side of the first
// interior cell: b += K_face * gamma * g (the outer row x_o = alpha x_q +
// gamma g eliminated from the fluid row). The BC rows' own right-hand side
// enters the stopping norm on the host. One launch for all faces and fields: a
// cell on several faces belongs to the first of them, whose thread adds the
// others' shares too (a launch per face and field was 18 launches per cavity
// step, 2.7 us each at 32^3).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kRiderThreads) k_bc_rhs(Geo g, OuterParams op, BcRhs p, SumRiders sums) {
    if ((int)blockIdx.z == p.nface) {
        if (blockIdx.x == 0 && blockIdx.y == 0) run_riders(sums);
        return;
    }
    const Dims &d = g.d;
    const int fc = p.face[blockIdx.z], ax = fc / 2, hi = fc % 2;
    const int n[3] = {d.nx, d.ny, d.nz};
    const int t1 = blockIdx.x * blockDim.x + threadIdx.x;
    const int t2 = blockIdx.y * blockDim.y + threadIdx.y;
    if (t1 >= (ax == 0 ? d.ny : d.nx) || t2 >= (ax == 2 ? d.ny : d.nz)) return;
    const int at = hi ? n[ax] - 1 : 0;
    const int i = ax == 0 ? at : t1, j = ax == 0 ? t1 : ax == 1 ? at : t2, k = ax == 2 ? at : t2;
    double v[3] = {0, 0, 0};
    for (int e = 0; e < p.nface; e++) {
        const int a = p.face[e] / 2, h = p.face[e] % 2;
        const int m = a == 0 ? i : a == 1 ? j : k;
        if (m != (h ? n[a] - 1 : 0)) continue;
        if (e < (int)blockIdx.z) return;  // an earlier face's cell
        const double kf = C1(p.K[a][h], m);
        for (int c = 0; c < p.n; c++)
            if (p.gamma[c][a][h] != 0)
                v[c] += kf * p.gamma[c][a][h]
                    * bcval(op.face[a][h], p.comp + c, a == 0 ? j : i, a == 2 ? j : k, a == 2 ? d.ny + 4 : d.nz);
    }
    const long q = cidx(d, i, j, k);
    for (int c = 0; c < p.n; c++) p.b[c][q] += v[c];
}

// ---------------------------------------------------------------------------
// Immersed-boundary ghost cells, ordered in-place update.
// <- src/ibm3d_fracstep.c:1933-1975. Ghost cells are grouped by dependency
// level; a source that is a ghost cell visited later in the reference's
// lexicographic order reads the value saved before the pass (old[]), one
// visited earlier reads the updated value (its level is lower).
// ---------------------------------------------------------------------------
// (the saving rides in the boundary layers' launch: save_ghosts)
__device__ inline void save_ghosts(const GhostSave &g, const OuterFields &fs) {
    const int t = threadIdx.x + blockDim.x * threadIdx.y, n = blockDim.x * blockDim.y;
    for (int s = (blockIdx.x + gridDim.x * blockIdx.y) * n + t; s < g.ng; s += gridDim.x * gridDim.y * n) {
        const long c = g.gc[s].cell;
        for (int e = 0; e < 4; e++) g.old[4 * (long)s + e] = fs.f[e][c];
    }
}

// Eight lanes per ghost cell, one per stencil point: bound by the chain of
// stencil entry, value and sum (one lane per cell: 8.7 us a level)
__device__ inline void ghost_cell(const GhostCell &G, const double *old, double *u1, double *u2, double *u3,
                                  double *p) {
    const int l = threadIdx.x & 7;
    const long c = G.src[l];
    double v[4] = {0, 0, 0, 0};
    if (c >= 0) {
        const double w = G.w[l];
        const int later = G.later[l];
        const double *f[4] = {u1, u2, u3, p};
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = w * (later >= 0 ? old[4 * (long)later + e] : f[e][c]);
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1)
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += __shfl_down(v[e], o, 8);
    if (l != 0) return;
    const double lu = 1 + G.wself, lp = 1 - G.wself;
    u1[G.cell] = -v[0] / lu;
    u2[G.cell] = -v[1] / lu;
    u3[G.cell] = -v[2] / lu;
    if (lp != 0) p[G.cell] = v[3] / lp;
}

__global__ void k_ghost_level(const GhostCell *gc, int s0, int s1, const double *old,
                              double *u1, double *u2, double *u3, double *p) {
    const int s = s0 + (blockIdx.x * blockDim.x + threadIdx.x) / 8;
    if (s < s1) ghost_cell(gc[s], old, u1, u2, u3, p);
}

// The small levels after it in one workgroup, a barrier between them
constexpr int kGhostTailThreads = 1024;
__global__ void __launch_bounds__(kGhostTailThreads) k_ghost_tail(const GhostCell *gc, GhostLevels lv,
                                                                  const double *old, double *u1, double *u2,
                                                                  double *u3, double *p) {
    for (int l = 0; l < lv.n; l++) {
        for (int s = lv.start[l] + threadIdx.x / 8; s < lv.start[l + 1]; s += kGhostTailThreads / 8)
            ghost_cell(gc[s], old, u1, u2, u3, p);
        __syncthreads();
    }
}

// Interior solid cells hold NaN in u and p (:1972-1973).
__global__ void k_solid_nan(Dims d, const uint8_t *flag, double *u1, double *u2, double *u3, double *p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= d.nx || j >= d.ny) return;
    const long q = cidx(d, i, j, k);
    if (flag[q] == F_SOLID) u1[q] = u2[q] = u3[q] = p[q] = nan_d();
}

// ---------------------------------------------------------------------------
// SGS stress.  <- src/ibm3d_turb.c:8-82 (Smagorinsky, l = min(Cs Delta,
// 0.41 phi), Delta = 2 cbrt(dx dy dz)); Vreman (extension) with
// nu_t = c sqrt(B / (alpha:alpha)). tau = -2 nu_t S on fluid cells only.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_sgs(Geo g, int model, double coef, VanDriest vd, const uint8_t *flag,
                                             const double *lvset, const double *u1, const double *u2,
                                             const double *u3, TauPtrs tau) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= d.nx || j >= d.ny) return;
    const long q = cidx(d, i, j, k);
    if (flag[q] != F_FLUID) return;
    const long sy = d.sy, sz = d.sz;
    const double ddx = C1(g.xc, i + 1) - C1(g.xc, i - 1);
    const double ddy = C1(g.yc, j + 1) - C1(g.yc, j - 1);
    const double ddz = C1(g.zc, k + 1) - C1(g.zc, k - 1);
    const double *uu[3] = {u1, u2, u3};
    double al[3][3];  // al[m][n] = d u_n / d x_m
#pragma unroll
    for (int n = 0; n < 3; n++) {
        al[0][n] = (uu[n][q + 1] - uu[n][q - 1]) / ddx;
        al[1][n] = (uu[n][q + sy] - uu[n][q - sy]) / ddy;
        al[2][n] = (uu[n][q + sz] - uu[n][q - sz]) / ddz;
    }
    // S in the reference's slot order 11, 12, 13, 22, 23, 33 (src/ibm3d_turb.c:60-81)
    double S[6];
    S[0] = al[0][0];
    S[1] = 0.5 * (al[1][0] + al[0][1]);
    S[2] = 0.5 * (al[2][0] + al[0][2]);
    S[3] = al[1][1];
    S[4] = 0.5 * (al[2][1] + al[1][2]);
    S[5] = al[2][2];
    double nut;
    if (model == 1) {
        const double delta = 2 * cbrt(C1(g.dx, i) * C1(g.dy, j) * C1(g.dz, k));
        // sum over all (a, b) of 2 S_ab^2, in the reference's loop order
        const double s2 = 2 * S[0] * S[0] + 2 * S[1] * S[1] + 2 * S[2] * S[2] + 2 * S[1] * S[1]
            + 2 * S[3] * S[3] + 2 * S[4] * S[4] + 2 * S[2] * S[2] + 2 * S[4] * S[4] + 2 * S[5] * S[5];
        const double smag = sqrt(s2);
        double l = coef * delta;
        if (vd.walls) {
            // van Driest: l *= 1 - exp(-y+ / A+), y+ = y_w u_tau / nu
            const double c[3] = {C1(g.xc, i), C1(g.yc, j), C1(g.zc, k)};
            const int bit_lo[3] = {8, 4, 16}, bit_hi[3] = {2, 1, 32};  // W S D, E N U
            double yw = 1e300;
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if (vd.walls & bit_lo[a]) yw = fmin(yw, c[a] - vd.lo[a]);
                if (vd.walls & bit_hi[a]) yw = fmin(yw, vd.hi[a] - c[a]);
            }
            l *= 1 - exp(-(yw * vd.ure) / vd.aplus);
        }
        const double lw = 0.41 * lvset[q];
        if (lw < l) l = lw;
        const double f = -2 * (l * l) * smag;
#pragma unroll
        for (int a = 0; a < 6; a++) tau.t[a][q] = f * S[a];
        return;
    }
    const double del[3] = {C1(g.dx, i), C1(g.dy, j), C1(g.dz, k)};
    double aa = 0, bt[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
            aa += al[a][b] * al[a][b];
            double acc = 0;
#pragma unroll
            for (int m = 0; m < 3; m++) acc += del[m] * del[m] * al[m][a] * al[m][b];
            bt[a][b] = acc;
        }
    const double Bb = bt[0][0] * bt[1][1] - bt[0][1] * bt[0][1] + bt[0][0] * bt[2][2] - bt[0][2] * bt[0][2]
        + bt[1][1] * bt[2][2] - bt[1][2] * bt[1][2];
    nut = (aa > 1e-300 && Bb > 0) ? coef * sqrt(Bb / aa) : 0;
#pragma unroll
    for (int a = 0; a < 6; a++) tau.t[a][q] = -2 * nut * S[a];
}

// max |div U| over fluid cells (partial maxima per block), the pinned cell
// (whose pressure row is the pin, not continuity) left out
__global__ void __launch_bounds__(256) k_maxdiv(Geo g, const uint8_t *flag, long pin, const double *U1,
                                                const double *U2, const double *U3, double *partial) {
    const Dims &d = g.d;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    double m = 0;
    if (i < d.nx && j < d.ny) {
        const long q = cidx(d, i, j, k);
        if (flag[q] == F_FLUID && q != pin) {
            const double v = (U1[q + 1] - U1[q]) / C1(g.dx, i) + (U2[q + d.sy] - U2[q]) / C1(g.dy, j)
                + (U3[q + d.sz] - U3[q]) / C1(g.dz, k);
            m = fabs(v);
        }
    }
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_down(m, o, 64));
    __shared__ double sh[16];
    const int tid = threadIdx.x + threadIdx.y * blockDim.x;
    if ((tid & 63) == 0) sh[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
        double r = 0;
        for (int w = 0; w < (int)((blockDim.x * blockDim.y + 63) / 64); w++) r = fmax(r, sh[w]);
        partial[block_linear()] = r;
    }
}

// Force on the immersed body (pressure and viscous parts, per unit density)
// from the staircase surface: the faces between an interior ghost cell and an
// interior fluid 6-neighbour, one thread per ghost cell. With n the outward
// body normal (from the ghost into the fluid cell) and A the face area:
//   pressure: F -= p_f n A, p_f linearly interpolated to the face position;
//   viscous:  F_b += mu (u_b(fluid) - u_b(ghost)) / |x_fluid - x_ghost| A for
//             the two tangential components b.
// No reference counterpart (the reference has no force diagnostic).
__global__ void __launch_bounds__(256) k_body_force(Geo g, const uint8_t *flag, const int *gijk, int ng, double mu,
                                                    const double *p, const double *u1, const double *u2,
                                                    const double *u3, double *partial) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    double f[3] = {0, 0, 0};
    if (t < ng) {
        const Dims &d = g.d;
        const int id[3] = {gijk[3 * t], gijk[3 * t + 1], gijk[3 * t + 2]};
        const long q = cidx(d, id[0], id[1], id[2]);
        const int n[3] = {d.nx, d.ny, d.nz};
        const long st[3] = {1, d.sy, d.sz};
        const double *C[3] = {g.xc, g.yc, g.zc}, *D[3] = {g.dx, g.dy, g.dz};
        const double *u[3] = {u1, u2, u3};
        const double h[3] = {C1(g.dx, id[0]), C1(g.dy, id[1]), C1(g.dz, id[2])};
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int sd = -1; sd <= 1; sd += 2) {
                const int nb = id[a] + sd;
                if (nb < 0 || nb >= n[a]) continue;
                const long r = q + sd * st[a];
                if (flag[r] != F_FLUID) continue;
                const double area = h[0] * h[1] * h[2] / h[a];
                const double xg = C1(C[a], id[a]), xf = C1(C[a], nb);
                const double xface = xg + sd * 0.5 * C1(D[a], id[a]);
                const double pf = p[q] + (p[r] - p[q]) * ((xface - xg) / (xf - xg));
                f[a] -= pf * sd * area;
                const double inv = 1.0 / fabs(xf - xg);
#pragma unroll
                for (int b = 0; b < 3; b++)
                    if (b != a) f[b] += mu * (u[b][r] - u[b][q]) * inv * area;
            }
    }
    block_sum_store<3>(f, partial, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Host layout (k fastest, src/utils.h:8-16) <-> device layout (i fastest),
// one (i, k) plane tile of 32 x 32 cells per block through LDS, so that both
// sides move whole lines. The transposition on the host walked one field
// plane-strided, a cache miss per element, after a copy of the whole padded
// allocation into a fresh host vector: 20 ms per field at 256 x 128 x 128,
// against 70 us here plus the copy of the reference layout itself.
// ---------------------------------------------------------------------------
constexpr int kRefTile = 32;
template <bool TO_HOST>
__global__ void __launch_bounds__(256) k_ref_layout(Dims d, double *f, double *ref, int ni, int nj, int nk, int i0,
                                                    int j0, int k0) {
    __shared__ double t[kRefTile][kRefTile + 1];
    const int ib = blockIdx.x * kRefTile, kb = blockIdx.y * kRefTile, j = blockIdx.z;
    const int tx = threadIdx.x, ty = threadIdx.y;
    if (TO_HOST) {
        for (int c = ty; c < kRefTile; c += 8)
            if (ib + tx < ni && kb + c < nk) t[c][tx] = f[cidx(d, i0 + ib + tx, j0 + j, k0 + kb + c)];
        __syncthreads();
        for (int a = ty; a < kRefTile; a += 8)
            if (ib + a < ni && kb + tx < nk) ref[((long)(ib + a) * nj + j) * nk + kb + tx] = t[tx][a];
    } else {
        for (int a = ty; a < kRefTile; a += 8)
            if (ib + a < ni && kb + tx < nk) t[tx][a] = ref[((long)(ib + a) * nj + j) * nk + kb + tx];
        __syncthreads();
        for (int c = ty; c < kRefTile; c += 8)
            if (ib + tx < ni && kb + c < nk) f[cidx(d, i0 + ib + tx, j0 + j, k0 + kb + c)] = t[c][tx];
    }
}

__global__ void __launch_bounds__(256) k_fill(double *a, long n, double v) {
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += 256L * gridDim.x) a[e] = v;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
void launch_ref_layout(hipStream_t st, const Dims &d, double *f, double *ref, int ni, int nj, int nk, int i0, int j0,
                       int k0, bool to_host) {
    const dim3 grid((ni + kRefTile - 1) / kRefTile, (nk + kRefTile - 1) / kRefTile, nj);
    if (to_host)
        hipLaunchKernelGGL(k_ref_layout<true>, grid, dim3(kRefTile, 8), 0, st, d, f, ref, ni, nj, nk, i0, j0, k0);
    else
        hipLaunchKernelGGL(k_ref_layout<false>, grid, dim3(kRefTile, 8), 0, st, d, f, ref, ni, nj, nk, i0, j0, k0);
}

void launch_fill(hipStream_t st, double *a, long n, double v) {
    const long nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(256), 0, st, a, n, v);
}

static dim3 cell_grid(const Dims &d, int ex) {
    return dim3((d.nx + ex + 63) / 64, (d.ny + ex + 3) / 4, d.nz + ex);
}

void launch_interp_stag(hipStream_t st, const Geo &g, const double *u1, const double *u2, const double *u3,
                        double *U1, double *U2, double *U3) {
    dim3 grid((g.d.nx + 4 + 63) / 64, (g.d.ny + 4 + 3) / 4, g.d.nz + 4);
    hipLaunchKernelGGL(k_interp_stag, grid, dim3(64, 4), 0, st, g, u1, u2, u3, U1, U2, U3);
}

long conv_rhs_blocks(const Dims &d) {
    dim3 gr = cell_grid(d, 0);
    return (long)gr.x * gr.y * gr.z;
}

void launch_conv_rhs(hipStream_t st, const Geo &g, const StepParams &sp, const uint8_t *flag,
                     const double *const u[3], const double *const U[3], const double *p,
                     const double *const Np[3], double *const N[3], double *const b[3], const TauPtrs &tau,
                     double *partial) {
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, cell_grid(g.d, 0), dim3(64, 4), 0, st, g, sp, flag, u[0], u[1], u[2], U[0], U[1],
                           U[2], p, Np[0], Np[1], Np[2], N[0], N[1], N[2], b[0], b[1], b[2], tau, partial);
    };
    if (sp.fa[0] || sp.fa[1] || sp.fa[2])
        tau.on ? launch(k_conv_rhs<true, true>) : launch(k_conv_rhs<false, true>);
    else
        tau.on ? launch(k_conv_rhs<true, false>) : launch(k_conv_rhs<false, false>);
}

void launch_face_star(hipStream_t st, const Geo &g, const StepParams &sp, const uint8_t *flag,
                      const double *const us[3], const double *p, double *const F[3]) {
    hipLaunchKernelGGL(k_face_star, cell_grid(g.d, 1), dim3(64, 4), 0, st, g, sp, flag, us[0], us[1], us[2],
                       p, F[0], F[1], F[2]);
}

void launch_poisson_rhs(hipStream_t st, const Geo &g, const StepParams &sp, const uint8_t *flag, long pin,
                        const double *const F[3], double *b, double *partial) {
    hipLaunchKernelGGL(k_poisson_rhs, cell_grid(g.d, 0), dim3(64, 4), 0, st, g, sp, flag, pin, F[0], F[1], F[2],
                       b, partial);
}

void launch_update(hipStream_t st, const Geo &g, const StepParams &sp, const uint8_t *flag, const double *p,
                   const double *pp, const double *const us[3], const double *const F[3], double *pn,
                   double *const un[3], double *const G[3]) {
    hipLaunchKernelGGL(k_update, cell_grid(g.d, 1), dim3(64, 4), 0, st, g, sp, flag, p, pp, us[0], us[1], us[2],
                       F[0], F[1], F[2], pn, un[0], un[1], un[2], G[0], G[1], G[2]);
}

void launch_outer(hipStream_t st, const Dims &d, const OuterParams &op, const OuterRule *rules,
                  const OuterFields &fs, const SumRiders &sums, const GhostSave &save) {
    const int m1 = std::max(d.ny, d.nx + 4), m2 = std::max(d.nz, d.ny + 4);
    const int nz = 12 * fs.n + (sums.n > 0 || save.ng > 0);
    hipLaunchKernelGGL(k_outer, dim3((m1 + 15) / 16, (m2 + 15) / 16, nz), dim3(16, 16), 0, st, d, op, rules, fs, sums,
                       save);
}

void launch_bc_rhs(hipStream_t st, const Geo &g, const OuterParams &op, const BcRhs &p, const SumRiders &sums) {
    const Dims &d = g.d;
    const int nz = p.nface + (sums.n > 0);
    if (nz == 0) return;
    const int m1 = p.nface ? std::max(d.nx, d.ny) : 1, m2 = p.nface ? std::max(d.ny, d.nz) : 1;
    hipLaunchKernelGGL(k_bc_rhs, dim3((m1 + 15) / 16, (m2 + 15) / 16, nz), dim3(16, 16), 0, st, g, op, p, sums);
}

// Largest number of cells of the levels that one workgroup takes: sphere 256 x
// 128 x 128, 1042 of 3568 cells in 6 levels, 37 us; level by level 10 us each. A
// tail of more cells goes on level by level.
constexpr int kGhostTail = 4096;

void launch_ghost_update(hipStream_t st, const GhostCell *gc, int ng, const int *level_start, int nlevels,
                         const double *old, double *u1, double *u2, double *u3, double *p) {
    for (int l = 0; l < nlevels; l++) {
        if (l > 0 && ng - level_start[l] <= kGhostTail && nlevels - l <= kGhostLevels) {
            GhostLevels lv{};
            for (; l < nlevels; l++) lv.start[lv.n++] = level_start[l];
            lv.start[lv.n] = level_start[nlevels];
            hipLaunchKernelGGL(k_ghost_tail, dim3(1), dim3(kGhostTailThreads), 0, st, gc, lv, old, u1, u2, u3, p);
            return;
        }
        const int s0 = level_start[l], s1 = level_start[l + 1];
        if (s1 > s0)
            hipLaunchKernelGGL(k_ghost_level, dim3((s1 - s0 + 31) / 32), dim3(256), 0, st, gc, s0, s1, old, u1, u2, u3,
                               p);
    }
}

void launch_solid_nan(hipStream_t st, const Dims &d, const uint8_t *flag, double *u1, double *u2, double *u3,
                      double *p) {
    hipLaunchKernelGGL(k_solid_nan, cell_grid(d, 0), dim3(64, 4), 0, st, d, flag, u1, u2, u3, p);
}

void launch_sgs(hipStream_t st, const Geo &g, int model, double coef, const VanDriest &vd, const uint8_t *flag,
                const double *lvset, const double *const u[3], const TauPtrs &tau) {
    hipLaunchKernelGGL(k_sgs, cell_grid(g.d, 0), dim3(64, 4), 0, st, g, model, coef, vd, flag, lvset, u[0], u[1],
                       u[2], tau);
}

long maxdiv_blocks(const Dims &d) { return conv_rhs_blocks(d); }

long body_force_blocks(int ng) { return (ng + 255) / 256 > 0 ? (ng + 255) / 256 : 1; }

void launch_body_force(hipStream_t st, const Geo &g, const uint8_t *flag, const int *gijk, int ng, double mu,
                       const double *p, const double *const u[3], double *partial) {
    hipLaunchKernelGGL(k_body_force, dim3(body_force_blocks(ng)), dim3(256), 0, st, g, flag, gijk, ng, mu, p, u[0],
                       u[1], u[2], partial);
}

void launch_maxdiv(hipStream_t st, const Geo &g, const uint8_t *flag, long pin, const double *const U[3],
                   double *partial) {
    hipLaunchKernelGGL(k_maxdiv, cell_grid(g.d, 0), dim3(64, 4), 0, st, g, flag, pin, U[0], U[1], U[2], partial);
}

}  // namespace ibm
