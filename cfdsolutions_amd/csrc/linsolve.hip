// Implicit-side kernels: approximate Roe Jacobian assembly into BSR, block
// SpMV, block ILU(0) and its triangular solves, block-Jacobi, the reference's
// block Gauss-Seidel and LU-SGS sweeps, and restarted FGMRES.
//
// Row-sequential algorithms (ILU(0), Gauss-Seidel, LU-SGS, triangular solves)
// follow the dependency DAG of the BSR pattern, a launch per level or rows
// handed over inside one launch (see "Row-to-row handover"): rows of one
// level do not depend on each other and every row performs the same
// operations in the same order as the sequential CPU code, so factors and
// sweeps are bit-identical to it.
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <vector>

#include "cfd_internal.h"

#include <type_traits>
#include "flux.h"

using namespace cfd;

namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// Jacobian blocks
// ---------------------------------------------------------------------------
// ConservativeEulerFluxJacobian, Euler3D/src/CompressibleUtils.cpp:558-609
__device__ __forceinline__ void flux_jac(double g, const double *Qc, double nx, double ny, double nz, double *J) {
    const double rho = Qc[0], u = Qc[1] / rho, v = Qc[2] / rho, w = Qc[3] / rho, rhoet = Qc[4];
    const double ek = 0.5 * (u * u + v * v + w * w);
    const double p = (g - 1.0) * (rhoet - rho * ek);
    const double ht = (rhoet + p) / rho;
    const double ubar = u * nx + v * ny + w * nz;
    J[0] = 0.0;
    J[5] = (g - 1.0) * ek * nx - u * ubar;
    J[10] = (g - 1.0) * ek * ny - v * ubar;
    J[15] = (g - 1.0) * ek * nz - w * ubar;
    J[20] = ((g - 1.0) * ek - ht) * ubar;
    J[1] = nx;
    J[6] = ubar - (g - 2.0) * u * nx;
    J[11] = v * nx - (g - 1.0) * u * ny;
    J[16] = w * nx - (g - 1.0) * u * nz;
    J[21] = ht * nx - (g - 1.0) * u * ubar;
    J[2] = ny;
    J[7] = u * ny - (g - 1.0) * v * nx;
    J[12] = ubar - (g - 2.0) * v * ny;
    J[17] = w * ny - (g - 1.0) * v * nz;
    J[22] = ht * ny - (g - 1.0) * v * ubar;
    J[3] = nz;
    J[8] = u * nz - (g - 1.0) * w * nx;
    J[13] = v * nz - (g - 1.0) * w * ny;
    J[18] = ubar - (g - 2.0) * w * nz;
    J[23] = ht * nz - (g - 1.0) * w * ubar;
    J[4] = 0.0;
    J[9] = (g - 1.0) * nx;
    J[14] = (g - 1.0) * ny;
    J[19] = (g - 1.0) * nz;
    J[24] = g * ubar;
}

// MC_Matrix_Mul_Matrix, MATH/src/MC_Iterative_Jacobi.c:192-207
__device__ __forceinline__ void mm5(const double *A, const double *B, double *C) {
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < 5; k++) s += A[5 * i + k] * B[5 * k + j];
            C[5 * i + j] = s;
        }
}

// Compute_RoeAJacobian, Euler3D/src/Roe_Fluxes.cpp:149-273: A = M P |Lambda| P^-1 M^-1
__device__ __forceinline__ void roe_ajac(double g, int efix, const double *QL, const double *QR, double nx, double ny,
                                         double nz, double *A) {
    Eos<double> L, R;
    eos_face(g, QL, nx, ny, nz, L);
    eos_face(g, QR, nx, ny, nz, R);
    const double rho = sqrt(R.rho * L.rho);
    const double sigma = rho / (L.rho + rho);
    const double u = L.u + sigma * (R.u - L.u);
    const double v = L.v + sigma * (R.v - L.v);
    const double w = L.w + sigma * (R.w - L.w);
    const double ht = L.ht + sigma * (R.ht - L.ht);
    const double c = roe_speed_sound(g, u, v, w, ht);
    const double ubar = u * nx + v * ny + w * nz;
    const double phi = 0.5 * (g - 1.0) * (u * u + v * v + w * w);
    const double M[25] = {1.0, 0.0, 0.0, 0.0, 0.0, u, rho, 0.0, 0.0, 0.0, v, 0.0, rho, 0.0, 0.0, w, 0.0, 0.0, rho, 0.0,
                          phi / (g - 1.0), rho * u, rho * v, rho * w, 1.0 / (g - 1.0)};
    const double Mi[25] = {1.0, 0.0, 0.0, 0.0, 0.0,
                           -u / rho, 1.0 / rho, 0.0, 0.0, 0.0,
                           -v / rho, 0.0, 1.0 / rho, 0.0, 0.0,
                           -w / rho, 0.0, 0.0, 1.0 / rho, 0.0,
                           phi, -u * (g - 1.0), -v * (g - 1.0), -w * (g - 1.0), (g - 1.0)};
    const double P[25] = {nx, ny, nz, rho / c, rho / c, 0.0, -nz, ny, nx, -nx, nz, 0.0, -nx, ny, -ny,
                          -ny, nx, 0.0, nz, -nz, 0.0, 0.0, 0.0, rho * c, rho * c};
    const double Pi[25] = {nx, 0.0, nz, -ny, -nx / (c * c),
                           ny, -nz, 0.0, nx, -ny / (c * c),
                           nz, ny, -nx, 0.0, -nz / (c * c),
                           0.0, 0.5 * nx, 0.5 * ny, 0.5 * nz, 1.0 / (2.0 * rho * c),
                           0.0, -0.5 * nx, -0.5 * ny, -0.5 * nz, 1.0 / (2.0 * rho * c)};
    double E0, E1, E2;
    roe_eigen(efix, L.ubar, L.c, R.ubar, R.c, ubar, c, E0, E1, E2);
    double T[25], Ti[25];
    mm5(M, P, T);
    mm5(Pi, Mi, Ti);
    // |Lambda| * Ti: the diagonal product of the reference's full multiply
    const double Ed[5] = {E0, E0, E0, E1, E2};
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) Ti[5 * i + j] = Ed[i] * Ti[5 * i + j];
    mm5(T, Ti, A);
}

template <class TA>
struct JacArgs {
    int N, NT;
    const int *order;
    const int *ip, *sptr, *nbr, *soff, *iau;
    const double *isx, *isy, *isz, *qa, *vol, *dt, *res;
    TA *a;
    double *b;
    double g;
    int efix, rhs_mode;
};

// Compute_Jacobian_Approximate_Roe, Euler3D/src/Roe_Jacobian.cpp:29-228,
// assembled by rows: node i writes its diagonal block (accumulated in edge
// order) and the off-diagonal block of every neighbour.
template <class TA>
__global__ __launch_bounds__(128) void k_jacobian(JacArgs<TA> a) {
    const int i = xcd_block() * 128 + threadIdx.x;  // internal node
    if (i >= a.N) return;
    const int ai = a.order[i];                      // its row of the BSR system
    double qi[5];
#pragma unroll
    for (int k = 0; k < 5; k++) qi[k] = a.qa[kQA * (size_t)i + k];
    double D[25];
#pragma unroll
    for (int t = 0; t < 25; t++) D[t] = 0.0;
    const double vd = a.vol[i] / a.dt[i];
#pragma unroll
    for (int t = 0; t < 5; t++) D[6 * t] = vd;
    const int deg = a.ip[i + 1] - a.ip[i];
    size_t idx = (size_t)a.sptr[i / kSlice] + (i % kSlice);
    for (int k = 0; k < deg; k++, idx += kSlice) {
        const int jr = ld_stream(a.nbr + idx);
        const bool iL = jr >= 0;  // ghosts (jr >= N) always pair with a physical L
        const int j = iL ? jr : ~jr;
        double nx, ny, nz;
        const double area = area_normal(ld_stream(a.isx + idx), ld_stream(a.isy + idx), ld_stream(a.isz + idx), nx,
                                        ny, nz);
        const double *rj = a.qa + kQA * (size_t)j;
        double QL[5], QR[5];
#pragma unroll
        for (int t = 0; t < 5; t++) {
            QL[t] = iL ? qi[t] : rj[t];
            QR[t] = iL ? rj[t] : qi[t];
        }
        double AR[25], J[25];
        roe_ajac(a.g, a.efix, QL, QR, nx, ny, nz, AR);
        if (j >= a.N) {
            flux_jac(a.g, QL, nx, ny, nz, J);
#pragma unroll
            for (int t = 0; t < 25; t++) D[t] += 0.5 * (J[t] + AR[t]) * area;
            continue;
        }
        TA *O = a.a + 25 * (size_t)ld_stream(a.soff + idx);
        if (iL) {
            flux_jac(a.g, QL, nx, ny, nz, J);
#pragma unroll
            for (int t = 0; t < 25; t++) D[t] += 0.5 * (J[t] + AR[t]) * area;
            flux_jac(a.g, QR, nx, ny, nz, J);
#pragma unroll
            for (int t = 0; t < 25; t++) O[t] = (TA)(0.0 + 0.5 * (J[t] - AR[t]) * area);
        } else {
            flux_jac(a.g, QR, nx, ny, nz, J);
#pragma unroll
            for (int t = 0; t < 25; t++) D[t] -= 0.5 * (J[t] - AR[t]) * area;
            flux_jac(a.g, QL, nx, ny, nz, J);
#pragma unroll
            for (int t = 0; t < 25; t++) O[t] = (TA)(0.0 - 0.5 * (J[t] + AR[t]) * area);
        }
    }
    TA *Dd = a.a + 25 * (size_t)a.iau[ai];
#pragma unroll
    for (int t = 0; t < 25; t++) Dd[t] = (TA)D[t];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        double r = a.res[kRES * (size_t)i + k];
        if (a.rhs_mode == 1) r = r + a.res[kRES * (size_t)i + 5 + k];
        a.b[5 * (size_t)ai + k] = -r;
    }
}

// Compute_RoeFlux, Euler3D/src/Roe_Fluxes.cpp:552-905 (Roe branch,
// conservative variables, no time term), returned as Conv + Diss per
// component: Conv = (F_L + F_R)|S|/2, Diss = -(M P |Lambda| P^-1 M^-1)(Q_R - Q_L)|S|/2.
__device__ __forceinline__ void roe_flux_matrix(double g, int efix, const double *QL, const double *QR, double sx,
                                                double sy, double sz, double *F) {
    double nx, ny, nz;
    const double area = area_normal(sx, sy, sz, nx, ny, nz);
    Eos<double> L, R;
    eos_face(g, QL, nx, ny, nz, L);
    eos_face(g, QR, nx, ny, nz, R);
    double fL[5], fR[5];
    fL[0] = L.rho * L.ubar;
    fL[1] = L.u * fL[0] + L.p * nx;
    fL[2] = L.v * fL[0] + L.p * ny;
    fL[3] = L.w * fL[0] + L.p * nz;
    fL[4] = L.ht * fL[0];
    fR[0] = R.rho * R.ubar;
    fR[1] = R.u * fR[0] + R.p * nx;
    fR[2] = R.v * fR[0] + R.p * ny;
    fR[3] = R.w * fR[0] + R.p * nz;
    fR[4] = R.ht * fR[0];
    double A[25];
    roe_ajac(g, efix, QL, QR, nx, ny, nz, A);
    double dQ[5];
#pragma unroll
    for (int t = 0; t < 5; t++) dQ[t] = QR[t] - QL[t];
#pragma unroll
    for (int r = 0; r < 5; r++) {
        double fa = 0.0;  // MC_Matrix_Mul_Vector
#pragma unroll
        for (int t = 0; t < 5; t++) fa += A[5 * r + t] * dQ[t];
        const double conv = 0.5 * (fL[r] + fR[r]) * area;
        const double diss = -0.5 * fa * area;
        F[r] = conv + diss;
    }
}

struct FdArgs {
    int N, NT;
    const int *order;
    const int *ip, *sptr, *nbr, *soff, *iau;
    const double *isx, *isy, *isz, *qa, *qb, *vol, *dt, *res;
    const int *btype, *bcase;
    const double *case_inf;
    double *a;
    float *af;
    double *b;
    double g, frac, coeff;
    int efix, rhs_mode, add_time, order2, lim, plus, minus, iter, zpg;
    BcFree<double> free;
    int *flag;
};

// Face states of an interior edge: Compute_SecondOrderReconstructQ
// (Euler3D/src/HigherOrderReconstructQ.cpp:20-71) for second order, the node
// values for first order.  o: this node, n: its neighbour, iL: this node is
// the L end.  Component c of the end `pend` (0 L, 1 R) is perturbed by dq if
// perturb is set.  All choices are selects, so nothing is indexed at run time.
struct FdNode {
    double q[5], x[3], g[15], p[5];
};

__device__ __forceinline__ void fd_faces(const FdArgs &a, const FdNode &o, const FdNode &n, bool iL, bool perturb,
                                         int pend, int c, double dq, double *QL, double *QR) {
    double qL[5], qR[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
        const double l = iL ? o.q[m] : n.q[m], r = iL ? n.q[m] : o.q[m];
        qL[m] = (perturb && pend == 0 && m == c) ? l + dq : l;
        qR[m] = (perturb && pend == 1 && m == c) ? r + dq : r;
    }
    if (!a.order2) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            QL[m] = qL[m];
            QR[m] = qR[m];
        }
        return;
    }
    const double xl0 = iL ? o.x[0] : n.x[0], xl1 = iL ? o.x[1] : n.x[1], xl2 = iL ? o.x[2] : n.x[2];
    const double xr0 = iL ? n.x[0] : o.x[0], xr1 = iL ? n.x[1] : o.x[1], xr2 = iL ? n.x[2] : o.x[2];
    const double RxL = 0.5 * (xr0 - xl0), RyL = 0.5 * (xr1 - xl1), RzL = 0.5 * (xr2 - xl2);
    const double RxR = -RxL, RyR = -RyL, RzR = -RzL;
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const double pL = a.lim ? (iL ? o.p[k] : n.p[k]) : 1.0, pR = a.lim ? (iL ? n.p[k] : o.p[k]) : 1.0;
        const double glx = iL ? o.g[3 * k] : n.g[3 * k], gly = iL ? o.g[3 * k + 1] : n.g[3 * k + 1],
                     glz = iL ? o.g[3 * k + 2] : n.g[3 * k + 2];
        const double grx = iL ? n.g[3 * k] : o.g[3 * k], gry = iL ? n.g[3 * k + 1] : o.g[3 * k + 1],
                     grz = iL ? n.g[3 * k + 2] : o.g[3 * k + 2];
        QL[k] = qL[k] + pL * (a.frac * (qR[k] - qL[k]) + (1.0 - a.frac) * (glx * RxL + gly * RyL + glz * RzL));
        QR[k] = qR[k] + pR * (a.frac * (qL[k] - qR[k]) + (1.0 - a.frac) * (grx * RxR + gry * RyR + grz * RzR));
    }
}

// Loads the record of node j: state, coordinates, and for second order the
// gradient and limiter.
__device__ __forceinline__ void fd_load(const FdArgs &a, int j, FdNode &r) {
    const double *ra = a.qa + kQA * (size_t)j;
#pragma unroll
    for (int m = 0; m < 5; m++) r.q[m] = ra[m];
#pragma unroll
    for (int m = 0; m < 3; m++) r.x[m] = ra[5 + m];
    if (a.order2 && j < a.N) {
        const double *rb = a.qb + kQB * (size_t)j;
#pragma unroll
        for (int f = 0; f < 15; f++) r.g[f] = rb[f];
#pragma unroll
        for (int m = 0; m < 5; m++) r.p[m] = rb[kPHI + m];
    } else {
#pragma unroll
        for (int f = 0; f < 15; f++) r.g[f] = 0.0;
#pragma unroll
        for (int m = 0; m < 5; m++) r.p[m] = 1.0;
    }
}

// The flux one finite-difference column differentiates: the matrix-form Roe
// flux (Compute_RoeFlux), or the scheme's own flux for HLLC and AUSM+ (the
// scheme-agnostic Compute_Jacobian_FiniteDifference,
// MPFLOW3D/src/FiniteDifference_Jacobian.cpp:112-667), whose dissipative
// part is zero.  F = conv + diss, as the oracle sums them.
template <int FLUX>
__device__ __forceinline__ void fd_edge_flux(const FdArgs &a, const double *QL, const double *QR, double sx, double sy,
                                             double sz, double *F) {
    if (FLUX == CFD_FLUX_ROE) {
        roe_flux_matrix(a.g, a.efix, QL, QR, sx, sy, sz, F);
        return;
    }
    double cf[5];
    int bad = 0;
    if (FLUX == CFD_FLUX_HLLC) hllc_flux(a.g, sx, sy, sz, QL, QR, cf, bad);
    else ausmp_flux(a.g, sx, sy, sz, QL, QR, cf);
    if (bad) atomicAdd(a.flag + 1, 1);
#pragma unroll
    for (int r = 0; r < 5; r++) F[r] = cf[r] + 0.0;
}

// Compute_Jacobian_FiniteDifference_Roe, Euler3D/src/Roe_Jacobian.cpp:236-776,
// assembled by rows with ten lanes per node: lane (role, c) walks the node's
// incidences in the reference's edge order and forms column c of
//   role 0: the derivative of each incident flux with respect to this node,
//           summed into the diagonal block (+ as L, - as R, then boundary
//           edges, central, ghost recomputed per perturbation);
//   role 1: the derivative with respect to the neighbour, written to the
//           off-diagonal block (0 + dF/dR as L, 0 - dF/dL as R).
// Each column costs two flux evaluations per incidence: perturbed +/- eps,
// or perturbed and unperturbed for the one-sided methods (the reference
// evaluates the unperturbed flux once per edge end and reuses it; the value
// is the same).
template <int FLUX>
__global__ __launch_bounds__(128) void k_jacobian_fd(FdArgs a) {
    const int t = blockIdx.x * 128 + threadIdx.x;
    const int i = t / 10;  // internal node
    if (i >= a.N) return;
    const int role = (t % 10) / 5, c = t % 5;
    const int ai = a.order[i];
    const double eps = 1.0E-8;
    FdNode own;
    fd_load(a, i, own);
    double D[5];  // column c of the diagonal block
#pragma unroll
    for (int r = 0; r < 5; r++) D[r] = (a.add_time && r == c) ? a.vol[i] / a.dt[i] : 0.0;
    const int deg = a.ip[i + 1] - a.ip[i];
    size_t idx = (size_t)a.sptr[i / kSlice] + (i % kSlice);
    for (int k = 0; k < deg; k++, idx += kSlice) {
        const int jr = ld_stream(a.nbr + idx);
        const bool iL = jr >= 0;  // ghosts (jr >= N) always pair with a physical L
        const int j = iL ? jr : ~jr;
        const double sx = ld_stream(a.isx + idx), sy = ld_stream(a.isy + idx), sz = ld_stream(a.isz + idx);
        if (j >= a.N) {  // boundary edge: central, this node perturbed
            if (role) continue;
            const int be = j - a.N;
            const double *rg = a.qa + kQA * (size_t)j;
            double qg[5];
#pragma unroll
            for (int m = 0; m < 5; m++) qg[m] = rg[m];
            const BcFree<double> fr = a.case_inf ? bc_free_of_case<double>(a.case_inf, a.bcase[be]) : a.free;
            double Fp[2][5];
#pragma unroll
            for (int pm = 0; pm < 2; pm++) {
                double QP[5], QG[5];
#pragma unroll
                for (int m = 0; m < 5; m++) QP[m] = (m == c) ? (pm ? own.q[m] - eps : own.q[m] + eps) : own.q[m];
                const int st = bc_ghost(a.g, QP, qg, sx, sy, sz, a.btype[be], a.iter, a.zpg, fr, QG);
                if (st == 2) {
                    atomicAdd(a.flag + 3, 1);
#pragma unroll
                    for (int m = 0; m < 5; m++) QG[m] = qg[m];
                } else if (st == 1) {
                    atomicAdd(a.flag + 0, 1);
                }
                fd_edge_flux<FLUX>(a, QP, QG, sx, sy, sz, Fp[pm]);
            }
#pragma unroll
            for (int r = 0; r < 5; r++) D[r] += 0.5 * (Fp[0][r] - Fp[1][r]) / eps;
            continue;
        }
        FdNode nb;
        fd_load(a, j, nb);
        // the perturbed end: this node (role 0) or the neighbour (role 1)
        const int pend = ((role == 0) == iL) ? 0 : 1;
        double FP[5], FM[5];
        {
            double QL[5], QR[5];
            fd_faces(a, own, nb, iL, a.plus, pend, c, eps, QL, QR);
            fd_edge_flux<FLUX>(a, QL, QR, sx, sy, sz, FP);
            fd_faces(a, own, nb, iL, a.minus, pend, c, -eps, QL, QR);
            fd_edge_flux<FLUX>(a, QL, QR, sx, sy, sz, FM);
        }
        double col[5];
#pragma unroll
        for (int r = 0; r < 5; r++) col[r] = a.coeff * (FP[r] - FM[r]) / eps;
        if (role == 0) {
#pragma unroll
            for (int r = 0; r < 5; r++) D[r] = iL ? D[r] + col[r] : D[r] - col[r];
        } else {
            const size_t o = 25 * (size_t)ld_stream(a.soff + idx) + c;
#pragma unroll
            for (int r = 0; r < 5; r++) {
                const double v = iL ? 0.0 + col[r] : 0.0 - col[r];
                if (a.af) a.af[o + 5 * r] = (float)v;
                else a.a[o + 5 * r] = v;
            }
        }
    }
    if (role == 0) {
        const size_t o = 25 * (size_t)a.iau[ai] + c;
#pragma unroll
        for (int r = 0; r < 5; r++) {
            if (a.af) a.af[o + 5 * r] = (float)D[r];
            else a.a[o + 5 * r] = D[r];
        }
        if (c == 0) {
#pragma unroll
            for (int k = 0; k < 5; k++) {
                double r = a.res[kRES * (size_t)i + k];
                if (a.rhs_mode == 1) r = r + a.res[kRES * (size_t)i + 5 + k];
                a.b[5 * (size_t)ai + k] = -r;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Dense 5x5 helpers (same operation order as the CPU oracle)
// ---------------------------------------------------------------------------
// Gauss-Jordan inverse with partial pivoting; returns false on a zero pivot.
// Every loop is unrolled and the pivot-row exchange is a select per entry, so
// the working matrix stays in registers (a dynamically indexed row swap put it
// in scratch memory); the arithmetic is the textbook sequence, unchanged.
__device__ bool inv5(const double *A, double *Ai) {
    double a[5][10];
#pragma unroll
    for (int r = 0; r < 5; r++)
#pragma unroll
        for (int c = 0; c < 5; c++) {
            a[r][c] = A[5 * r + c];
            a[r][c + 5] = (r == c) ? 1.0 : 0.0;
        }
#pragma unroll
    for (int c = 0; c < 5; c++) {
        // first row of largest magnitude in column c (ties keep the earlier row)
        int piv = c;
        double best = fabs(a[c][c]);
#pragma unroll
        for (int r = c + 1; r < 5; r++) {
            const double v = fabs(a[r][c]);
            if (v > best) {
                piv = r;
                best = v;
            }
        }
#pragma unroll
        for (int r = c + 1; r < 5; r++) {
            const bool sw = piv == r;
#pragma unroll
            for (int j = 0; j < 10; j++) {
                const double t = a[c][j];
                a[c][j] = sw ? a[r][j] : t;
                a[r][j] = sw ? t : a[r][j];
            }
        }
        const double d = a[c][c];
        if (d == 0.0) return false;
#pragma unroll
        for (int j = 0; j < 10; j++) a[c][j] = a[c][j] / d;
#pragma unroll
        for (int r = 0; r < 5; r++) {
            if (r == c) continue;
            const double f = a[r][c];
#pragma unroll
            for (int j = 0; j < 10; j++) a[r][j] = a[r][j] - f * a[c][j];
        }
    }
#pragma unroll
    for (int r = 0; r < 5; r++)
#pragma unroll
        for (int c = 0; c < 5; c++) Ai[5 * r + c] = a[r][c + 5];
    return true;
}

// ---------------------------------------------------------------------------
// Block ILU(0), the rows of one level: Saad Alg. 10.4 in block form, the
// operations of orc_ilu0 on every entry in its order.  Factors in TM; the
// pivot inverse is computed in FP64.
//
// Up to kIluFewRows rows (k_ilu0_level) G groups of five lanes share a block
// row, 12 / G rows to a wavefront: lane r of group g holds row r of the row's
// blocks g, g + G, ... in registers from the first load to the store (blocks
// past the kIluSets of a lane stay in lu, read and written by the lane that owns
// them; the columns of the next NX are in registers, a row still longer is
// searched for each of row k's columns).  For the lower block (i, k) every group forms L_ik = A_ik D_k^-1 for
// itself, finds which of row k's upper columns its own blocks have, and
// subtracts L_ik U_kj; the updates of one k run side by side.  Such a level's
// time is that of one row's chain over its lower blocks.  With a row's blocks in
// memory and one group per row, a level of the 48x16x16 mesh took 46 us (FP64,
// natural order) and 72 us (FP32, multicolour), now 16.6 and 24 us.
//
// Wider levels (k_ilu0_rows) are bound by instructions and by the reads of row
// k's blocks: five lanes to a row, 12 rows to a wavefront, each lane's row of
// the blocks in an LDS column of its own.  Colours of 95,000 rows on average:
// 401 us with three rows to a wavefront as above, now 253 (FP32, 763k rows in 8
// colours); of 102,000 rows 739, now 523 us (FP64).  A row's blocks are read in
// flights of five: waiting for each cost 30 us a colour.  Reading the next
// pivot's blocks and the next update's ahead spilled and lost (384 us).
// ---------------------------------------------------------------------------
// One row per wavefront up to kIluNarrowRows (four wavefronts per SIMD): at
// 1,770 rows of a level 24 us against 30 us with three rows, at 5,700 44 us
// against 35 us (FP32).  Three rows up to kIluFewRows: at 6,800 rows 33 us
// against 37 us with 12 rows, at 13,300 65 us against 53 us.
//
// Rows of unstructured meshes are longer and differ in length (Delaunay meshes:
// 16.5 blocks on average, up to 70), so rows that share a wavefront wait for
// the longest, and blocks past 15 stay in memory in k_ilu0_rows.  There
// (cfd_mesh::ilu_long) one row per wavefront is ahead at every width in FP32
// and up to kIluLongRows rows in FP64.  Delaunay meshes, multicolour, whole
// factorisation, ms in FP64 / FP32, with the lines of short rows and as it is:
// 60,000 rows 3.45 / 3.05 and 2.7 / 2.2; 200,000 rows 9.1 / 7.3 and 7.9 / 5.7;
// 500,000 rows 14.7 / 11.1 and 14.6 / 10.1.
constexpr int kIluNarrowRows = 4096, kIluFewRows = 8192, kIluLongRows = 32768;
template <int G>
constexpr int kIluSets = (16 + G - 1) / G;

// The slot of the row's blocks [b0, b1) that has column c, or -1 (ascending
// columns).
__device__ __forceinline__ int find_col(const int *__restrict__ ja, int b0, int b1, int c) {
    const int end = b1;
    while (b0 < b1) {
        const int mid = b0 + (b1 - b0) / 2;
        if (ja[mid] < c) b0 = mid + 1;
        else b1 = mid;
    }
    return b0 < end && ja[b0] == c ? b0 : -1;
}

// Row r of a block in memory loses L U (r: row of L).
template <class TM>
__device__ __forceinline__ void block_update(TM *B, const TM *L, const TM *__restrict__ U) {
    TM u[25];
#pragma unroll
    for (int z = 0; z < 25; z++) u[z] = U[z];
#pragma unroll
    for (int c = 0; c < 5; c++) {
        TM v = TM(0.0);
#pragma unroll
        for (int z = 0; z < 5; z++) v += L[z] * u[5 * z + c];
        B[c] = B[c] - v;
    }
}

// MORE: rows may have blocks that stay in lu (2 to 4% of the time where none has).
template <class TM, int G, bool MORE>
__global__ __launch_bounds__(kBlock) void k_ilu0_level(int nrows, const int *__restrict__ rows,
                                                      const int *__restrict__ ia, const int *__restrict__ ja,
                                                      const int *__restrict__ iau, const int *__restrict__ src,
                                                      const TM *__restrict__ a, TM *lu, TM *dinv,
                                                      const TM *__restrict__ luk, const TM *__restrict__ dinvk,
                                                      int *flag) {
    // luk / dinvk view the blocks and inverse pivots of rows of earlier
    // levels, which this launch only reads (it writes rows of one level).
    // src: slot of A for each slot of the pattern (NULL: the same).
    constexpr int NS = kIluSets<G>, NX = 24 / G, RW = 12 / G, W = 5 * G;
    __shared__ double diag[kBlock / 64][RW][25];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rs = lane / W, base = rs * W, in = lane - base, g = in / 5, r = in - 5 * g;
    const int t = (blockIdx.x * (kBlock / 64) + wave) * RW + rs;
    const bool active = rs < RW && t < nrows;
    const int i = active ? rows[t] : 0;
    const int b0 = active ? ia[i] : 0, n = active ? ia[i + 1] - b0 : 0, nl = active ? iau[i] - b0 : 0;
    int col[NS], up[NS], nu[NS];  // the blocks' columns; for lower ones the upper blocks of that row
    TM T[NS][5];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int b = s * G + g;
        col[s] = -1;
        up[s] = nu[s] = 0;
        if (b < n) {
            col[s] = ja[b0 + b];
            const TM *A = a + 25 * (size_t)(src ? src[b0 + b] : b0 + b) + 5 * r;
#pragma unroll
            for (int c = 0; c < 5; c++) T[s][c] = A[c];
            if (b < nl) {
                up[s] = iau[col[s]] + 1;
                nu[s] = ia[col[s] + 1] - up[s];
            }
        }
    }
    const bool more = MORE && __any(n > NS * G);  // a row has blocks that stay in lu: the columns of the next NX per lane
    int xcol[NX];
    if (more) {
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int b = (NS + x) * G + g;
            xcol[x] = b < n ? ja[b0 + b] : -1;
        }
        for (int b = NS * G + g; b < n; b += G) {
            const TM *A = a + 25 * (size_t)(src ? src[b0 + b] : b0 + b) + 5 * r;
            for (int c = 0; c < 5; c++) lu[25 * (size_t)(b0 + b) + 5 * r + c] = A[c];
        }
    }
    for (int l = 0; __any(l < nl); l++) {
        const int so = l / G, from = base + 5 * (l - so * G);
        int k = 0, p0 = 0, np = 0;
        TM Ar[5] = {};
#pragma unroll
        for (int s = 0; s < NS; s++)
            if (so == s) {
                k = __shfl(col[s], from, 64);
                p0 = __shfl(up[s], from, 64);
                np = __shfl(nu[s], from, 64);
#pragma unroll
                for (int c = 0; c < 5; c++) Ar[c] = __shfl(T[s][c], from + r, 64);
            }
        if (so >= NS) {
            for (int c = 0; c < 5; c++) {
                if (l < nl && 5 * g == from - base) Ar[c] = lu[25 * (size_t)(b0 + l) + 5 * r + c];
                Ar[c] = __shfl(Ar[c], from + r, 64);
            }
            if (l < nl) {
                k = ja[b0 + l];
                p0 = iau[k] + 1;
                np = ia[k + 1] - p0;
            }
        }
        if (l >= nl) continue;
        TM D[25], L[5];
#pragma unroll
        for (int q = 0; q < 25; q++) D[q] = dinvk[25 * (size_t)k + q];
        // which of row k's upper blocks meets each of this lane's blocks; eight
        // columns at a time (ja is padded by kIluPad entries)
        int hit[NS], xhit[NX];
#pragma unroll
        for (int s = 0; s < NS; s++) hit[s] = -1;
#pragma unroll
        for (int x = 0; x < NX; x++) xhit[x] = -1;
        for (int c0 = 0; c0 < np; c0 += kIluPad) {
            int cq[kIluPad];
#pragma unroll
            for (int q = 0; q < kIluPad; q++) cq[q] = ja[p0 + c0 + q];
#pragma unroll
            for (int q = 0; q < kIluPad; q++)
#pragma unroll
                for (int s = 0; s < NS; s++) hit[s] = ((cq[q] == col[s]) & (c0 + q < np)) ? c0 + q : hit[s];
            if (more)
#pragma unroll
                for (int q = 0; q < kIluPad; q++)
#pragma unroll
                    for (int x = 0; x < NX; x++) xhit[x] = ((cq[q] == xcol[x]) & (c0 + q < np)) ? c0 + q : xhit[x];
        }
#pragma unroll
        for (int c = 0; c < 5; c++) {
            TM s = TM(0.0);
#pragma unroll
            for (int q = 0; q < 5; q++) s += Ar[q] * D[5 * q + c];
            L[c] = s;
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (s * G + g == l) {
#pragma unroll
                for (int c = 0; c < 5; c++) T[s][c] = L[c];
            } else if (hit[s] >= 0) {
                const TM *U = luk + 25 * (size_t)(p0 + hit[s]);
                TM u[25];
#pragma unroll
                for (int q = 0; q < 25; q++) u[q] = U[q];
#pragma unroll
                for (int c = 0; c < 5; c++) {
                    TM v = TM(0.0);
#pragma unroll
                    for (int q = 0; q < 5; q++) v += L[q] * u[5 * q + c];
                    T[s][c] = T[s][c] - v;
                }
            }
        }
        if (!more) continue;
        TM *const row = lu + 25 * (size_t)b0 + 5 * r;
        if (l >= NS * G && l % G == g)
            for (int c = 0; c < 5; c++) row[25 * (size_t)l + c] = L[c];
#pragma unroll
        for (int x = 0; x < NX; x++)
            if (xhit[x] >= 0) block_update(row + 25 * (size_t)((NS + x) * G + g), L, luk + 25 * (size_t)(p0 + xhit[x]));
        const int t0 = max((NS + NX) * G, l + 1);  // the blocks past those, sought from row k's side
        for (int q = 0; t0 < n && q < np; q++) {
            const int b = find_col(ja, b0 + t0, b0 + n, ja[p0 + q]) - b0;
            if (b >= t0 && b % G == g) block_update(row + 25 * (size_t)b, L, luk + 25 * (size_t)(p0 + q));
        }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int b = s * G + g;
        if (b >= n) continue;
        TM *B = lu + 25 * (size_t)(b0 + b) + 5 * r;
#pragma unroll
        for (int c = 0; c < 5; c++) {
            B[c] = T[s][c];
            if (b == nl) diag[wave][rs][5 * r + c] = (double)T[s][c];
        }
    }
    for (int b = NS * G + g; b < n; b += G)
        if (b == nl)
            for (int c = 0; c < 5; c++) diag[wave][rs][5 * r + c] = (double)lu[25 * (size_t)(b0 + b) + 5 * r + c];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // Gauss-Jordan inverse of inv5 with one column of [D | I] to a lane (the
    // row's first ten lanes): the same operations on every entry
    double m[5];
#pragma unroll
    for (int q = 0; q < 5; q++)
        m[q] = !active ? 0.0 : in < 5 ? diag[wave][rs][5 * q + in] : (in - 5 == q ? 1.0 : 0.0);
    bool singular = false;
#pragma unroll
    for (int c = 0; c < 5; c++) {
        double p[5];
#pragma unroll
        for (int q = 0; q < 5; q++) p[q] = __shfl(m[q], base + c, 64);
        int piv = c;
        double best = fabs(p[c]);
#pragma unroll
        for (int q = c + 1; q < 5; q++) {
            const double v = fabs(p[q]);
            if (v > best) {
                piv = q;
                best = v;
            }
        }
#pragma unroll
        for (int q = c + 1; q < 5; q++) {
            const bool sw = piv == q;
            const double x = m[c], y = p[c];
            m[c] = sw ? m[q] : x;
            m[q] = sw ? x : m[q];
            p[c] = sw ? p[q] : y;
            p[q] = sw ? y : p[q];
        }
        singular = singular || p[c] == 0.0;
        m[c] = m[c] / p[c];
#pragma unroll
        for (int q = 0; q < 5; q++)
            if (q != c) m[q] = m[q] - p[q] * m[c];
    }
    if (!active) return;
    if (singular && in == 0) atomicAdd(flag + 2, 1);
    if (in >= 5 && in < 10)
#pragma unroll
        for (int q = 0; q < 5; q++) dinv[25 * (size_t)i + 5 * q + in - 5] = singular ? TM(0.0) : (TM)m[q];
}

// The same factorisation with five lanes to a block row, 12 rows to a
// wavefront: lane r keeps row r of the blocks in its own LDS column, where the
// block that an update meets can be looked up, so L_ik is formed once, the rows'
// searches are shared out (lane r compares the columns of blocks r, r + 5, ...)
// and a row's updates follow each other without idle lanes.
constexpr int kIluCols = kIluKeep / 5;                           // blocks of a row kept in LDS, the rest stay in lu:
constexpr int kIluMore = 4, kIluSeen = kIluKeep + 5 * kIluMore;  // of these so many have their columns in registers

template <class TM, bool MORE>
__global__ __launch_bounds__(64) void k_ilu0_rows(int nrows, const int *__restrict__ rows, const int *__restrict__ ia,
                                                  const int *__restrict__ ja, const int *__restrict__ iau,
                                                  const int *__restrict__ src, const TM *__restrict__ a, TM *lu,
                                                  TM *dinv, const TM *__restrict__ luk, const TM *__restrict__ dinvk,
                                                  int *flag) {
    __shared__ TM keep[kIluKeep][5][60];
    __shared__ double diag[12][25];
    const int lane = threadIdx.x, rs = lane / 5, base = 5 * rs, r = lane - base;
    const int t = blockIdx.x * 12 + rs;
    const bool active = rs < 12 && t < nrows;
    const int i = active ? rows[t] : 0;
    const int b0 = active ? ia[i] : 0, n = active ? ia[i + 1] - b0 : 0, nl = active ? iau[i] - b0 : 0;
    int col[kIluCols], up[kIluCols], nu[kIluCols];  // of blocks r, r + 5, ..; for lower ones the upper blocks of that row
#pragma unroll
    for (int s = 0; s < kIluCols; s++) {
        const int b = 5 * s + r;
        col[s] = -1;
        up[s] = nu[s] = 0;
        if (b < n) {
            col[s] = ja[b0 + b];
            if (b < nl) {
                up[s] = iau[col[s]] + 1;
                nu[s] = ia[col[s] + 1] - up[s];
            }
        }
    }
    // all reads in flight at once: past the row's end its last block again
    int sl[kIluKeep];
#pragma unroll
    for (int b = 0; b < kIluKeep; b++) {
        const int q = b0 + max(0, min(b, n - 1));
        sl[b] = src ? src[q] : q;
    }
    for (int h = 0; h < kIluCols; h++) {
        TM A[5][5];
#pragma unroll
        for (int b = 0; b < 5; b++)
#pragma unroll
            for (int c = 0; c < 5; c++)
                A[b][c] = a[25 * (size_t)(h == 0 ? sl[b] : h == 1 ? sl[b + 5] : sl[b + 10]) + 5 * r + c];
        if (lane < 60)
#pragma unroll
            for (int b = 0; b < 5; b++)
#pragma unroll
                for (int c = 0; c < 5; c++) keep[5 * h + b][c][lane] = A[b][c];
    }
    const bool more = MORE && __any(n > kIluKeep);
    int xcol[kIluMore];
    if (more) {
#pragma unroll
        for (int x = 0; x < kIluMore; x++) {
            const int b = kIluKeep + 5 * x + r;
            xcol[x] = b < n ? ja[b0 + b] : -1;
        }
        for (int b = kIluKeep; b < n; b++) {
            const TM *A = a + 25 * (size_t)(src ? src[b0 + b] : b0 + b) + 5 * r;
            for (int c = 0; c < 5; c++) lu[25 * (size_t)(b0 + b) + 5 * r + c] = A[c];
        }
    }
    for (int l = 0; l < nl; l++) {  // (the lanes of a row stay together)
        int k, p0, np;
        TM Ar[5], L[5], D[25];
        if (l < kIluKeep) {
            const int so = l / 5, from = base + l - 5 * so;
            k = __shfl(so == 0 ? col[0] : so == 1 ? col[1] : col[2], from, 64);
            p0 = __shfl(so == 0 ? up[0] : so == 1 ? up[1] : up[2], from, 64);
            np = __shfl(so == 0 ? nu[0] : so == 1 ? nu[1] : nu[2], from, 64);
#pragma unroll
            for (int c = 0; c < 5; c++) Ar[c] = keep[l][c][lane];
        } else {
            k = ja[b0 + l];
            p0 = iau[k] + 1;
            np = ia[k + 1] - p0;
            for (int c = 0; c < 5; c++) Ar[c] = lu[25 * (size_t)(b0 + l) + 5 * r + c];
        }
#pragma unroll
        for (int q = 0; q < 25; q++) D[q] = dinvk[25 * (size_t)k + q];
        int hit[kIluCols], xhit[kIluMore];
#pragma unroll
        for (int s = 0; s < kIluCols; s++) hit[s] = -1;
#pragma unroll
        for (int x = 0; x < kIluMore; x++) xhit[x] = -1;
        for (int c0 = 0; c0 < np; c0 += kIluPad) {  // (ja is padded by kIluPad entries)
            int cq[kIluPad];
#pragma unroll
            for (int q = 0; q < kIluPad; q++) cq[q] = ja[p0 + c0 + q];
#pragma unroll
            for (int q = 0; q < kIluPad; q++)
#pragma unroll
                for (int s = 0; s < kIluCols; s++) hit[s] = ((cq[q] == col[s]) & (c0 + q < np)) ? c0 + q : hit[s];
            if (more)
#pragma unroll
                for (int q = 0; q < kIluPad; q++)
#pragma unroll
                    for (int x = 0; x < kIluMore; x++)
                        xhit[x] = ((cq[q] == xcol[x]) & (c0 + q < np)) ? c0 + q : xhit[x];
        }
        unsigned mask = 0;  // blocks of the row that row k's upper blocks meet
#pragma unroll
        for (int s = 0; s < kIluCols; s++) mask |= (unsigned)(__ballot(hit[s] >= 0) >> base & 31) << (5 * s);
#pragma unroll
        for (int c = 0; c < 5; c++) {
            TM v = TM(0.0);
#pragma unroll
            for (int q = 0; q < 5; q++) v += Ar[q] * D[5 * q + c];
            L[c] = v;
        }
        if (l < kIluKeep) {
#pragma unroll
            for (int c = 0; c < 5; c++) keep[l][c][lane] = L[c];
        } else {
            for (int c = 0; c < 5; c++) lu[25 * (size_t)(b0 + l) + 5 * r + c] = L[c];
        }
        for (; mask; mask &= mask - 1) {
            const int b = __ffs(mask) - 1, so = b / 5;
            const int q = __shfl(so == 0 ? hit[0] : so == 1 ? hit[1] : hit[2], base + b - 5 * so, 64);
            const TM *U = luk + 25 * (size_t)(p0 + q);
            TM u[25];
#pragma unroll
            for (int z = 0; z < 25; z++) u[z] = U[z];
#pragma unroll
            for (int c = 0; c < 5; c++) {
                TM v = TM(0.0);
#pragma unroll
                for (int z = 0; z < 5; z++) v += L[z] * u[5 * z + c];
                keep[b][c][lane] = keep[b][c][lane] - v;
            }
        }
        if (!more) continue;
        TM *const row = lu + 25 * (size_t)b0 + 5 * r;
        unsigned xmask = 0;  // the same of the blocks in lu
#pragma unroll
        for (int x = 0; x < kIluMore; x++) xmask |= (unsigned)(__ballot(xhit[x] >= 0) >> base & 31) << (5 * x);
        for (; xmask; xmask &= xmask - 1) {
            const int b = __ffs(xmask) - 1, so = b / 5;
            const int q = __shfl(so == 0 ? xhit[0] : so == 1 ? xhit[1] : so == 2 ? xhit[2] : xhit[3], base + b - 5 * so, 64);
            block_update(row + 25 * (size_t)(kIluKeep + b), L, luk + 25 * (size_t)(p0 + q));
        }
        const int t0 = max(kIluSeen, l + 1);  // the blocks past those, sought from row k's side
        for (int q = 0; t0 < n && q < np; q++) {
            const int b = find_col(ja, b0 + t0, b0 + n, ja[p0 + q]) - b0;
            if (b >= t0) block_update(row + 25 * (size_t)b, L, luk + 25 * (size_t)(p0 + q));
        }
    }
#pragma unroll
    for (int b = 0; b < kIluKeep; b++)
        if (b < n) {
            TM *B = lu + 25 * (size_t)(b0 + b) + 5 * r;
#pragma unroll
            for (int c = 0; c < 5; c++) B[c] = keep[b][c][lane];
        }
    if (active)
        for (int c = 0; c < 5; c++)
            diag[rs][5 * r + c] =
                (double)(nl < kIluKeep ? keep[nl][c][lane] : lu[25 * (size_t)(b0 + nl) + 5 * r + c]);
    __syncthreads();
    // Gauss-Jordan inverse of inv5, columns r of D and of I to a lane: the same
    // operations on every entry
    double m[5], w[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        m[q] = active ? diag[rs][5 * q + r] : 0.0;
        w[q] = r == q ? 1.0 : 0.0;
    }
    bool singular = false;
#pragma unroll
    for (int c = 0; c < 5; c++) {
        double p[5];
#pragma unroll
        for (int q = 0; q < 5; q++) p[q] = __shfl(m[q], base + c, 64);
        int piv = c;
        double best = fabs(p[c]);
#pragma unroll
        for (int q = c + 1; q < 5; q++) {
            const double v = fabs(p[q]);
            if (v > best) {
                piv = q;
                best = v;
            }
        }
#pragma unroll
        for (int q = c + 1; q < 5; q++) {
            const bool sw = piv == q;
            const double x = m[c], y = p[c], z = w[c];
            m[c] = sw ? m[q] : x;
            m[q] = sw ? x : m[q];
            p[c] = sw ? p[q] : y;
            p[q] = sw ? y : p[q];
            w[c] = sw ? w[q] : z;
            w[q] = sw ? z : w[q];
        }
        singular = singular || p[c] == 0.0;
        m[c] = m[c] / p[c];
        w[c] = w[c] / p[c];
#pragma unroll
        for (int q = 0; q < 5; q++)
            if (q != c) {
                m[q] = m[q] - p[q] * m[c];
                w[q] = w[q] - p[q] * w[c];
            }
    }
    if (!active) return;
    if (singular && r == 0) atomicAdd(flag + 2, 1);
#pragma unroll
    for (int q = 0; q < 5; q++) dinv[25 * (size_t)i + 5 * q + r] = singular ? TM(0.0) : (TM)w[q];
}

// Inverse diagonal blocks (block-Jacobi).
template <class TA, class TM>
__global__ __launch_bounds__(kBlock) void k_block_inv(int N, const int *iau, const TA *a, TM *dinv, int *flag) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    double Dg[25], Di[25];
    for (int q = 0; q < 25; q++) Dg[q] = (double)a[25 * (size_t)iau[i] + q];
    if (!inv5(Dg, Di)) {
        atomicAdd(flag + 2, 1);
        for (int q = 0; q < 25; q++) Di[q] = 0.0;
    }
    for (int q = 0; q < 25; q++) dinv[25 * (size_t)i + q] = (TM)Di[q];
}

// Triangular solves of ILU(0), one level; 5 lanes per row (lane r owns
// component r).  Forward: z_i = r_i - sum_{k<i} L_ik z_k.  Backward:
// z_i = D_i^-1 (z_i - sum_{k>i} U_ik z_k).
template <class TM, class TV>
__global__ __launch_bounds__(kBlock) void k_trsv_level(int nrows, const int *__restrict__ rows,
                                                       const int *__restrict__ ia, const int *__restrict__ ja,
                                                       const int *__restrict__ iau, const TM *__restrict__ lu,
                                                       const TM *__restrict__ dinv, const TV *__restrict__ rhs, TV *z,
                                                       int backward) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int slot = lane / 5, r = lane - 5 * slot;
    const int t = (blockIdx.x * (kBlock / 64) + wave) * 12 + slot;
    const bool active = slot < 12 && t < nrows;
    const int i = active ? rows[t] : 0;
    TV y = TV(0.0);
    if (active) {
        if (!backward) {
            y = rhs[5 * (size_t)i + r];
            for (int kk = ia[i]; kk < iau[i]; kk++) {
                const TM *A = lu + 25 * (size_t)kk + 5 * r;
                const TV *zj = z + 5 * (size_t)ja[kk];
                TV s = TV(0.0);
#pragma unroll
                for (int c = 0; c < 5; c++) s += (TV)A[c] * zj[c];
                y = y - s;
            }
        } else {
            y = z[5 * (size_t)i + r];
            for (int kk = iau[i] + 1; kk < ia[i + 1]; kk++) {
                const TM *A = lu + 25 * (size_t)kk + 5 * r;
                const TV *zj = z + 5 * (size_t)ja[kk];
                TV s = TV(0.0);
#pragma unroll
                for (int c = 0; c < 5; c++) s += (TV)A[c] * zj[c];
                y = y - s;
            }
        }
    }
    if (!backward) {
        if (active) z[5 * (size_t)i + r] = y;
        return;
    }
    // gather the row's 5 components from its lanes, then apply D_i^-1
    const int base = lane - r;
    TV yy[5];
#pragma unroll
    for (int c = 0; c < 5; c++) yy[c] = __shfl(y, base + c, 64);
    if (active) {
        const TM *D = dinv + 25 * (size_t)i + 5 * r;
        TV s = TV(0.0);
#pragma unroll
        for (int c = 0; c < 5; c++) s += (TV)D[c] * yy[c];
        z[5 * (size_t)i + r] = s;
    }
}

// ---------------------------------------------------------------------------
// Row-to-row handover: sweeps whose rows depend on one another run in one
// launch, each row starting as soon as the rows it reads are done.
//
// A value and the fact that it is ready are one aligned word: every word of
// the handover array holds a NaN with a payload of its own ("unset") until its
// row stores the result, so a reader needs no flag, no fence and no ordering
// between addresses.  The 8 XCDs' L2s are not coherent with one another, so
// both sides use relaxed agent-scope accesses, which go past them.  (A flag per
// row needs a release store, which writes the XCD's L2 back: 1244 us per FP64
// sweep over the 14,161 rows in 205 levels of the 48x16x16 mesh, 6 us a level;
// one word per value: 354 us.)  A result that is itself a NaN is stored as the
// default NaN, so no result can look unset.
//
// Rows go in chunks of 12 in level order (levels are padded to whole chunks),
// so a chunk reads only earlier ones.  A running wave or workgroup draws its next
// chunks by a ticket when it is done with the last: the earliest unfinished
// chunk is always held by a wave that runs, whatever else the GPU holds and
// however many of the launch's workgroups it holds, so a wait always ends.  (A
// fixed share of the chunks to each workgroup needs every workgroup resident.)
// A wait over cfd_mesh::spin_max polls (a word beside the flags) raises flag[3],
// and every waiter gives up once it is set: a sweep ends even where a store is
// lost, and the solve reports it.
//
// flow_blocks: how many workgroups pay depends on how many chunks can run at a
// time (a level's).  Too few leave loads unissued, too many poll more than they
// work.  Twenty Arnoldi steps, ms at 128, 256 and 512 workgroups: 6 chunks
// (48x16x16, natural order, FP64) 15.0, 15.6, 17.2; 33 (120x40x40) 41.8, 42.8,
// 50.0; 81 (192x64x64) 82.2, 79.8, 97.3; 147 (48x16x16, colours) 2.06, 1.96,
// 2.16; 333 (Delaunay mesh of 60,000, colours) -, 7.2, 7.8; 475 (72x24x24,
// colours) 4.80, 3.24, 3.18; 1,088 (95x33x31, colours) -, 6.3, 5.5.
// ---------------------------------------------------------------------------
inline int flow_blocks(const cfd_mesh *m, int64_t chunks, int64_t width) {
    const int64_t n = m->flow_blocks ? m->flow_blocks : width < 60 ? 128 : width < 400 ? 256 : 512;
    return (int)std::min((chunks + 3) / 4, n);
}

template <class T>
struct FlowWord;
template <>
struct FlowWord<double> {
    using U = unsigned long long;
    static constexpr U unset = 0x7ff8c0ded15ea5edull, nan = 0x7ff8000000000000ull;
};
template <>
struct FlowWord<float> {
    using U = unsigned;
    static constexpr U unset = 0x7fc5a17du, nan = 0x7fc00000u;
};

template <class T>
__device__ __forceinline__ T ld_coh(const T *p) {
    return __hip_atomic_load(const_cast<T *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void st_coh(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ typename FlowWord<T>::U flow_load(const T *p) {
    return ld_coh(reinterpret_cast<const typename FlowWord<T>::U *>(p));
}
template <class T>
__device__ __forceinline__ void flow_store(T *p, T v) {
    using W = FlowWord<T>;
    st_coh(reinterpret_cast<typename W::U *>(p), v == v ? __builtin_bit_cast(typename W::U, v) : W::nan);
}
template <class T>
__device__ __forceinline__ void flow_unset(T *p) {
    st_coh(reinterpret_cast<typename FlowWord<T>::U *>(p), FlowWord<T>::unset);
}
// Whether poll `it` of a wait was its last: the bound is reached or another
// wait's was.
__device__ __forceinline__ bool flow_give_up(int it, int *flag) {
    if ((it & 255) != 255 || (it < ld_coh(flag + kFlagSpin) && ld_coh(flag + 3) == 0)) return false;
    atomicOr(flag + 3, 1);
    return true;
}
// The value of word p, of which v has been read already.
template <class T>
__device__ __forceinline__ T flow_wait(const T *p, typename FlowWord<T>::U v, int *flag) {
    for (int it = 0; v == FlowWord<T>::unset && !flow_give_up(it, flag); it++) v = flow_load(p);
    return __builtin_bit_cast(T, v);
}

// A wave's next chunk, from the launch's counter.  It is drawn when the last
// chunk is done: the answer to a ticket drawn ahead is waited for with the
// chunk's own loads, which are answered in order (20 Gauss-Seidel sweeps of the
// 48x16x16 mesh 2.4 against 1.7 ms).
__device__ __forceinline__ int flow_ticket(int *count) {
    int w = 0;
    if ((threadIdx.x & 63) == 0) w = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_amdgcn_readfirstlane(w);
}
// The same for a workgroup's four waves at once, where a launch's many short
// chunks would crowd the counter (colours of 104,448 rows: 20 Arnoldi steps 5.5
// ms, 8.3 with a ticket to a wave; Gauss-Seidel sweeps, with more work to a
// chunk, lose by the barrier: 1.7 against 1.4 ms): for (w = next();
// more(total); w = next()), with nothing to do for a wave whose w is not below
// total.
struct FlowGroup {
    int *const count, *const shared;  // the counter, two words of LDS
    int n = 0;
    __device__ __forceinline__ FlowGroup(int *c, int *s) : count(c), shared(s) {}
    __device__ __forceinline__ int next() {
        n ^= 1;
        if (threadIdx.x == 0)
            shared[n] = (kBlock / 64) * __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        return __builtin_amdgcn_readfirstlane(shared[n] + (int)(threadIdx.x >> 6));
    }
    __device__ __forceinline__ bool more(int total) const { return __builtin_amdgcn_readfirstlane(shared[n]) < total; }
};

// Also sets a launch's ticket counter back (NULL: none).
template <class T>
__global__ __launch_bounds__(kBlock) void k_flow_unset(size_t n, T *x, int *ticket) {
    if (ticket && blockIdx.x == 0 && threadIdx.x == 0) st_coh(ticket, 0);
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) flow_unset(x + i);
}

// One to U blocks of a row at once, without branches: places
// past the last block repeat it, and their products are dropped.  Lane r of the
// row's five loads row r of every block and component r of every neighbour, all
// before the wait, so that the entries are there when the last neighbour
// arrives; the neighbours' components then go through LDS to the other lanes.
// (What a row costs after its last neighbour is mostly instructions of one
// wave: with a branch, a wait and shuffles per block the FP64 sweep of the
// 48x16x16 mesh took 685 us, with one wait for all blocks 400 us, so 354 us;
// the handover itself takes 0.4 us of a level's 1.7 us.)
template <class T>
struct FlowLds {
    static constexpr int row = sizeof(T) == 8 ? 6 : 8;     // values of a neighbour (5), aligned for wide reads
    static constexpr int slot = 8 * row + (sizeof(T) == 8 ? 2 : 4);  // rows of a wavefront start in different banks
    T v[kBlock / 64][13 * slot];
};
template <int U, class TM, class TV>
struct FlowBlocks {
    TM av[U][5];
    const TV *x;  // component r of row 0
    int j[U], n;
    typename FlowWord<TV>::U v[U];
    __device__ __forceinline__ void load(int k0, int ke, int r, const int *__restrict__ ja, const TM *__restrict__ a,
                                         const TV *xx) {
        x = xx + r;
        n = ke - k0;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = u < n ? k0 + u : ke - 1;
            j[u] = ja[k];
            v[u] = flow_load(x + 5 * (size_t)j[u]);
#pragma unroll
            for (int c = 0; c < 5; c++) av[u][c] = a[25 * (size_t)k + 5 * r + c];
        }
    }
    // Waits until every neighbour is there: all words are read again together
    // until none is unset, so the row goes on one read after its last
    // neighbour's store (one word after the other costs a read, 0.4 us, each).
    __device__ __forceinline__ void wait(int *flag) {
        for (int it = 0;; it++) {
            bool all = true;
#pragma unroll
            for (int u = 0; u < U; u++) all = all & (v[u] != FlowWord<TV>::unset);
            if (all) return;
            if (flow_give_up(it, flag)) return;
#pragma unroll
            for (int u = 0; u < U; u++)
                if (v[u] == FlowWord<TV>::unset) v[u] = flow_load(x + 5 * (size_t)j[u]);
        }
    }
    __device__ __forceinline__ void share(TV *sh, int r) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < U; u++) sh[u * FlowLds<TV>::row + r] = __builtin_bit_cast(TV, v[u]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // s plus the products one after the other, as k_spmv adds them.
    __device__ __forceinline__ TV add_dots(TV *sh, int r, TV s) {
        share(sh, r);
#pragma unroll
        for (int u = 0; u < U; u++) {
            TV q = s;
#pragma unroll
            for (int c = 0; c < 5; c++) q += (TV)av[u][c] * sh[u * FlowLds<TV>::row + c];
            s = u < n ? q : s;
        }
        return s;
    }
    // t[u] = (row r of block u) . (neighbour u); sh: this row's place in LDS.
    __device__ __forceinline__ void dots(TV *sh, int r, TV *t) {
        share(sh, r);
#pragma unroll
        for (int u = 0; u < U; u++) {
            TV s = TV(0.0);
#pragma unroll
            for (int c = 0; c < 5; c++) s += (TV)av[u][c] * sh[u * FlowLds<TV>::row + c];
            t[u] = u < n ? s : TV(0.0);
        }
    }
};

// The ILU(0) apply and the product that follows it in an Arnoldi step, in one
// launch; 12 rows of 5 lanes per wavefront, lane r owns component r.  Items, in
// the order the wavefronts take them:
//   forward    w_i = r_P(i) - sum_{k<i} L_ik w_k, r = V_j, here also normalised and
//              stored from the last step's w where norm2 is given (k_scale_dev)
//   backward   z_P(i) = w_i = D_i^-1 (w_i - sum_{k>i} U_ik w_k)
//   product    y_i = sum_k A_ik z_k
// in the operation order of k_trsv_level, k_trsv_mc and k_spmv.  P is the row
// permutation perm of the multicolour order (NULL: the natural order); A is in
// the reference's order.  Handover words: of the forward sweep, the backward
// sweep and (where P is given) of z in the reference's order.  The other set of
// words is left unset for the next launch, so nothing is cleared while it is
// read.  A backward row starts when its own neighbours are done, a product
// while the last rows still run, and four launches are saved.
template <class TM, class TV>
struct FlowStep {
    int nf, nb, np;          // padded rows of the sweeps' schedules, rows of the product (0: none)
    const int *sf, *sb;      // the schedules
    const int *ia, *ja, *iau, *perm;
    const TM *lu, *dinv;
    const TV *w;             // last step's w (norm2) or unused
    const double *norm2;     // its squared norm, or NULL
    TV *v, *z, *y;           // V_j, Z_j, the product
    const int *aia, *aja;
    const TM *a;
    TV *words, *other;       // this launch's set of handover words and the next one's
    size_t L;
    int *flag, *ticket, *next_ticket;  // this launch's counter and the next one's, set back here
};

template <class TM>
constexpr int kTrsvPerCu = sizeof(TM) == 4 ? 4 : 2;
template <class TM, class TV>
__global__ __launch_bounds__(kBlock, kTrsvPerCu<TM>) void k_arnoldi_flow(FlowStep<TM, TV> f) {
    const int lane = threadIdx.x & 63, slot = lane / 5, r = lane - 5 * slot, base = lane - r;
    TV *wf = f.words, *wb = f.words + f.L, *wz = f.perm ? wb + f.L : wb;
    __shared__ __align__(16) FlowLds<TV> lds;
    TV *sh = lds.v[threadIdx.x >> 6] + slot * FlowLds<TV>::slot;
    const double denom = f.norm2 ? sqrt(f.norm2[0]) : 1.0;
    const int cf = (f.nf + 11) / 12, cb = (f.nb + 11) / 12, cp = (f.np + 11) / 12;
    __shared__ int tickets[2];
    FlowGroup q(f.ticket, tickets);
    const int total = cf + cb + cp;
    for (int w = q.next(); q.more(total); w = q.next()) {
        if (w == 0 && lane == 0) st_coh(f.next_ticket, 0);
        if (w >= total) continue;
        FlowBlocks<8, TM, TV> g;
        if (w >= cf + cb) {
            const int i = 12 * (w - cf - cb) + slot;
            if (slot < 12 && i < f.np) {
                const int ke = f.aia[i + 1];
                TV s = TV(0.0);
                for (int k0 = f.aia[i]; k0 < ke; k0 += 8) {
                    g.load(k0, ke, r, f.aja, f.a, wz);
                    g.wait(f.flag);
                    s = g.add_dots(sh, r, s);
                }
                f.y[5 * (size_t)i + r] = s;
            }
            continue;
        }
        const bool backward = w >= cf;
        TV *cur = backward ? wb : wf;
        const int t = 12 * (backward ? w - cf : w) + slot;
        const int i = slot < 12 && t < (backward ? f.nb : f.nf) ? (backward ? f.sb : f.sf)[t] : -1;
        const size_t ri = 5 * (size_t)(i >= 0 ? i : 0) + r;
        TV y = TV(0.0);
        TM dr[5];
        size_t pi = 0;
        if (i >= 0) {
            pi = 5 * (size_t)(f.perm ? f.perm[i] : i) + r;
            const int kb = backward ? f.iau[i] + 1 : f.ia[i];
            const int ke = backward ? f.ia[i + 1] : f.iau[i];
            if (backward) {
#pragma unroll
                for (int c = 0; c < 5; c++) dr[c] = f.dinv[25 * (size_t)i + 5 * r + c];
                y = flow_wait(wf + ri, flow_load(wf + ri), f.flag);
            } else {
                y = f.norm2 ? (TV)((double)f.w[pi] / denom) : f.v[pi];
                if (f.norm2) f.v[pi] = y;
                flow_unset(f.other + ri);
                flow_unset(f.other + f.L + ri);
                if (f.perm) flow_unset(f.other + 2 * f.L + ri);
            }
            for (int k0 = kb; k0 < ke; k0 += 8) {
                TV t8[8];
                g.load(k0, ke, r, f.ja, f.lu, cur);
                g.wait(f.flag);
                g.dots(sh, r, t8);
#pragma unroll
                for (int u = 0; u < 8; u++) y = y - t8[u];
            }
        }
        if (backward) {
            // gather the row's 5 components from its lanes, then apply D_i^-1
            TV yy[5];
#pragma unroll
            for (int c = 0; c < 5; c++) yy[c] = __shfl(y, base + c, 64);
            if (i >= 0) {
                TV s = TV(0.0);
#pragma unroll
                for (int c = 0; c < 5; c++) s += (TV)dr[c] * yy[c];
                y = s;
                f.z[pi] = y;
                if (f.perm) flow_store(wz + pi, y);
            }
        }
        if (i >= 0) flow_store(cur + ri, y);
    }
}

// One level of the multicolour ILU(0) sweeps; rows and columns are in
// multicolour order, the right-hand side and the result in the reference
// order (perm maps a multicolour row to its reference row).  Forward:
// w_i = r_perm(i) - sum_{k<i} L_ik w_k.  Backward: w_i = D_i^-1 (w_i -
// sum_{k>i} U_ik w_k), z_perm(i) = w_i.  5 lanes per row, as k_trsv_level.
template <class TM, class TV>
__global__ __launch_bounds__(kBlock) void k_trsv_mc(int nrows, const int *__restrict__ rows,
                                                    const int *__restrict__ ia, const int *__restrict__ ja,
                                                    const int *__restrict__ iau, const int *__restrict__ perm,
                                                    const TM *__restrict__ lu, const TM *__restrict__ dinv,
                                                    const TV *__restrict__ rhs, TV *w, TV *z, int backward) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int slot = lane / 5, r = lane - 5 * slot;
    const int t = (blockIdx.x * (kBlock / 64) + wave) * 12 + slot;
    const bool active = slot < 12 && t < nrows;
    const int i = active ? rows[t] : 0;
    TV y = TV(0.0);
    if (active) {
        const int kb = backward ? iau[i] + 1 : ia[i];
        const int ke = backward ? ia[i + 1] : iau[i];
        y = backward ? w[5 * (size_t)i + r] : rhs[5 * (size_t)perm[i] + r];
        // four blocks at a time: their loads are all issued before the
        // products are subtracted, in block order as one at a time
        for (int k0 = kb; k0 < ke; k0 += 4) {
            int jj[4];
#pragma unroll
            for (int u = 0; u < 4; u++) jj[u] = k0 + u < ke ? ja[k0 + u] : -1;
            TM av[4][5];
            TV wv[4][5];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (jj[u] >= 0) {
#pragma unroll
                    for (int c = 0; c < 5; c++) {
                        av[u][c] = lu[25 * (size_t)(k0 + u) + 5 * r + c];
                        wv[u][c] = w[5 * (size_t)jj[u] + c];
                    }
                }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (jj[u] >= 0) {
                    TV s = TV(0.0);
#pragma unroll
                    for (int c = 0; c < 5; c++) s += (TV)av[u][c] * wv[u][c];
                    y = y - s;
                }
        }
    }
    if (!backward) {
        if (active) w[5 * (size_t)i + r] = y;
        return;
    }
    const int base = lane - r;
    TV yy[5];
#pragma unroll
    for (int c = 0; c < 5; c++) yy[c] = __shfl(y, base + c, 64);
    if (active) {
        const TM *D = dinv + 25 * (size_t)i + 5 * r;
        TV s = TV(0.0);
#pragma unroll
        for (int c = 0; c < 5; c++) s += (TV)D[c] * yy[c];
        w[5 * (size_t)i + r] = s;
        z[5 * (size_t)perm[i] + r] = s;
    }
}

// One colour of the multicolour ILU(0) sweeps with the factors in block-SELL
// layout: rows r0..r1-1 (permuted order, one colour, independent of each
// other), one row per lane.  Forward: w_i = r_P(i) - sum over the strict lower
// blocks L_ij w_j; backward: w_i = D_i^-1 (w_i - sum over the strict upper
// blocks U_ij w_j), also scattered to z in original order.  Same operation
// order as k_trsv_mc.  Workgroups are numbered XCD by XCD (the grid is a
// multiple of the XCD count), so each XCD sweeps a contiguous range of the
// colour's rows and gathers from fewer lines of w.
template <class TM, class TV>
__global__ __launch_bounds__(kBlock) void k_trsv_mc_sell(int r0, int r1, const int *__restrict__ ia,
                                                         const int *__restrict__ iau, const int *__restrict__ perm,
                                                         const int *__restrict__ off, const int *__restrict__ col,
                                                         const TM *__restrict__ val, const TM *__restrict__ dv,
                                                         const TV *__restrict__ rhs, TV *w, TV *z, int backward) {
    const int i = (r0 & ~63) + xcd_block() * kBlock + threadIdx.x;
    if (i < r0 || i >= r1) return;
    const int l = i & 63;
    const int len = backward ? ia[i + 1] - iau[i] - 1 : iau[i] - ia[i];
    TV y[5];
#pragma unroll
    for (int r = 0; r < 5; r++) y[r] = backward ? w[5 * (size_t)i + r] : rhs[5 * (size_t)perm[i] + r];
    // U blocks at a time: their column indices, then their x values and
    // entries (streamed: each is read once per sweep) are loaded before the
    // products, which are then subtracted in block order as before.
    constexpr int U = sizeof(TM) == 8 ? 2 : 4;
    size_t p = (size_t)off[i >> 6] + l;
    for (int k0 = 0; k0 < len; k0 += U, p += 64 * U) {
        int jj[U];
#pragma unroll
        for (int u = 0; u < U; u++) jj[u] = k0 + u < len ? col[p + 64 * u] : -1;
        TV wv[U][5];
        TM av[U][25];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (jj[u] >= 0) {
                const TV *wj = w + 5 * (size_t)jj[u];
#pragma unroll
                for (int c = 0; c < 5; c++) wv[u][c] = wj[c];
                const TM *A = val + 25 * (p + 64 * u - l) + l;
#pragma unroll
                for (int e = 0; e < 25; e++) av[u][e] = ld_stream(A + 64 * e);
            }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (jj[u] >= 0) {
#pragma unroll
                for (int r = 0; r < 5; r++) {
                    TV s = TV(0.0);
#pragma unroll
                    for (int c = 0; c < 5; c++) s += (TV)av[u][5 * r + c] * wv[u][c];
                    y[r] = y[r] - s;
                }
            }
    }
    if (!backward) {
#pragma unroll
        for (int r = 0; r < 5; r++) w[5 * (size_t)i + r] = y[r];
        return;
    }
    const TM *D = dv + 25 * (size_t)(i - l) + l;
#pragma unroll
    for (int r = 0; r < 5; r++) {
        TV s = TV(0.0);
#pragma unroll
        for (int c = 0; c < 5; c++) s += (TV)D[64 * (5 * r + c)] * y[c];
        w[5 * (size_t)i + r] = s;
        z[5 * (size_t)perm[i] + r] = s;
    }
}

// FP16 block-SELL copy of FP32 blocks: each block's 25 entries over its
// largest magnitude (a zero block keeps scale 1), the scale kept per slot.
__global__ __launch_bounds__(kBlock) void k_to_sell_half(size_t nblk, const int *__restrict__ src,
                                                         const float *__restrict__ v, _Float16 *__restrict__ out,
                                                         float *__restrict__ scale) {
    for (size_t p = blockIdx.x * (size_t)kBlock + threadIdx.x; p < nblk; p += (size_t)gridDim.x * kBlock) {
        const int q = src ? src[p] : (int)p;
        if (q < 0) continue;
        const size_t l = p & 63;
        _Float16 *o = out + 25 * (p - l) + l;
        const float *in = v + 25 * (size_t)q;
        float mx = 0.0f;
#pragma unroll
        for (int e = 0; e < 25; e++) mx = fmaxf(mx, fabsf(in[e]));
        const float sc = mx > 0.0f ? mx : 1.0f, inv = 1.0f / sc;
#pragma unroll
        for (int e = 0; e < 25; e++) o[64 * e] = (_Float16)(in[e] * inv);
        scale[p] = sc;
    }
}

// k_trsv_mc_sell with the factors stored in FP16 (per-block FP32 scales):
// each block's product is formed in FP32 and scaled once.
__global__ __launch_bounds__(kBlock) void k_trsv_mc_sell_half(int r0, int r1, const int *__restrict__ ia,
                                                              const int *__restrict__ iau, const int *__restrict__ perm,
                                                              const int *__restrict__ off, const int *__restrict__ col,
                                                              const _Float16 *__restrict__ val,
                                                              const float *__restrict__ vsc,
                                                              const _Float16 *__restrict__ dv,
                                                              const float *__restrict__ dsc,
                                                              const float *__restrict__ rhs, float *w, float *z,
                                                              int backward) {
    const int i = (r0 & ~63) + xcd_block() * kBlock + threadIdx.x;
    if (i < r0 || i >= r1) return;
    const int l = i & 63;
    const int len = backward ? ia[i + 1] - iau[i] - 1 : iau[i] - ia[i];
    float y[5];
#pragma unroll
    for (int r = 0; r < 5; r++) y[r] = backward ? w[5 * (size_t)i + r] : rhs[5 * (size_t)perm[i] + r];
    constexpr int U = 4;  // blocks whose loads are in flight together, as in k_trsv_mc_sell
    size_t p = (size_t)off[i >> 6] + l;
    for (int k0 = 0; k0 < len; k0 += U, p += 64 * U) {
        int jj[U];
#pragma unroll
        for (int u = 0; u < U; u++) jj[u] = k0 + u < len ? col[p + 64 * u] : -1;
        float wv[U][5], sc[U];
        _Float16 av[U][25];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (jj[u] >= 0) {
                const float *wj = w + 5 * (size_t)jj[u];
#pragma unroll
                for (int c = 0; c < 5; c++) wv[u][c] = wj[c];
                const _Float16 *A = val + 25 * (p + 64 * u - l) + l;
#pragma unroll
                for (int e = 0; e < 25; e++) av[u][e] = ld_stream(A + 64 * e);
                sc[u] = ld_stream(vsc + p + 64 * u);
            }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (jj[u] >= 0) {
#pragma unroll
                for (int r = 0; r < 5; r++) {
                    float s = 0.0f;
#pragma unroll
                    for (int c = 0; c < 5; c++) s += (float)av[u][5 * r + c] * wv[u][c];
                    y[r] = y[r] - sc[u] * s;
                }
            }
    }
    if (!backward) {
#pragma unroll
        for (int r = 0; r < 5; r++) w[5 * (size_t)i + r] = y[r];
        return;
    }
    const _Float16 *D = dv + 25 * (size_t)(i - l) + l;
    const float sd = dsc[i];
#pragma unroll
    for (int r = 0; r < 5; r++) {
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < 5; c++) s += (float)D[64 * (5 * r + c)] * y[c];
        s *= sd;
        w[5 * (size_t)i + r] = s;
        z[5 * (size_t)perm[i] + r] = s;
    }
}

// z = D^-1 r (block-Jacobi apply)
template <class TM, class TV>
__global__ __launch_bounds__(kBlock) void k_bjac_apply(int N, const TM *dinv, const TV *rhs, TV *z) {
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= 5 * N) return;
    const int i = t / 5, r = t - 5 * i;
    const TM *D = dinv + 25 * (size_t)i + 5 * r;
    const TV *x = rhs + 5 * (size_t)i;
    TV s = TV(0.0);
#pragma unroll
    for (int c = 0; c < 5; c++) s += (TV)D[c] * x[c];
    z[t] = s;
}

// y = A x, one thread per (row, component); sum over blocks then columns.
template <class TA, class TX, class TY>
__global__ __launch_bounds__(kBlock) void k_spmv(int N, const int *__restrict__ ia, const int *__restrict__ ja,
                                                 const TA *__restrict__ a, const TX *__restrict__ x, TY *__restrict__ y,
                                                 const double *__restrict__ bsub) {
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= 5 * N) return;
    const int i = t / 5, r = t - 5 * i;
    TY s = TY(0.0);
    // four blocks at a time (loads first, then the products in order)
    const int ke = ia[i + 1];
    for (int k0 = ia[i]; k0 < ke; k0 += 4) {
        int jj[4];
#pragma unroll
        for (int u = 0; u < 4; u++) jj[u] = k0 + u < ke ? ja[k0 + u] : -1;
        TA av[4][5];
        TX xv[4][5];
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (jj[u] >= 0) {
#pragma unroll
                for (int c = 0; c < 5; c++) {
                    av[u][c] = a[25 * (size_t)(k0 + u) + 5 * r + c];
                    xv[u][c] = x[5 * (size_t)jj[u] + c];
                }
            }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (jj[u] >= 0) {
#pragma unroll
                for (int c = 0; c < 5; c++) s += (TY)av[u][c] * (TY)xv[u][c];
            }
    }
    if (bsub) s = (TY)bsub[t] - s;  // residual form r = b - A x
    y[t] = s;
}

// Copies BSR-ordered blocks (25 values each) into a block-SELL layout: slot
// p takes block src[p]; padding slots are left as they are (never read).
template <class T>
__global__ __launch_bounds__(kBlock) void k_to_sell(size_t nblk, const int *__restrict__ src, const T *__restrict__ v,
                                                    T *__restrict__ out) {
    for (size_t p = blockIdx.x * (size_t)kBlock + threadIdx.x; p < nblk; p += (size_t)gridDim.x * kBlock) {
        const int q = src ? src[p] : (int)p;
        if (q < 0) continue;
        const size_t l = p & 63;
        T *o = out + 25 * (p - l) + l;
        const T *in = v + 25 * (size_t)q;
#pragma unroll
        for (int e = 0; e < 25; e++) o[64 * e] = in[e];
    }
}

// y = A x (or y = b - A x) with A in block-SELL layout, one row per lane.  Each
// row's sum runs over its blocks in BSR order and each block's columns in
// order, as k_spmv and the oracle add them, so the bits are the same.  Rows
// go to the XCDs in contiguous ranges (grid a multiple of the XCD count) and
// the entries, read once per product, are streamed past the L2.
template <class TA, class TX, class TY>
__global__ __launch_bounds__(kBlock) void k_spmv_sell(int N, const int *__restrict__ ia, const int *__restrict__ off,
                                                      const int *__restrict__ col, const TA *__restrict__ val,
                                                      const TX *__restrict__ x, TY *__restrict__ y,
                                                      const double *__restrict__ bsub) {
    const int i = xcd_block() * kBlock + threadIdx.x;
    if (i >= N) return;
    const int l = i & 63;
    const int len = ia[i + 1] - ia[i];
    size_t p = (size_t)off[i >> 6] + l;
    TY s[5];
#pragma unroll
    for (int r = 0; r < 5; r++) s[r] = TY(0.0);
    for (int k = 0; k < len; k++, p += 64) {
        const TX *xj = x + 5 * (size_t)col[p];
        TX xv[5];
#pragma unroll
        for (int c = 0; c < 5; c++) xv[c] = xj[c];
        const TA *A = val + 25 * (p - l) + l;
#pragma unroll
        for (int r = 0; r < 5; r++)
#pragma unroll
            for (int c = 0; c < 5; c++) s[r] += (TY)ld_stream(A + 64 * (5 * r + c)) * (TY)xv[c];
    }
#pragma unroll
    for (int r = 0; r < 5; r++) {
        TY v = s[r];
        if (bsub) v = (TY)bsub[5 * (size_t)i + r] - v;  // residual form r = b - A x
        y[5 * (size_t)i + r] = v;
    }
}

// k_spmv_sell with A stored in FP16 (per-block FP32 scales): each block's
// product is formed in FP32 and scaled once.
template <class TX, class TY>
__global__ __launch_bounds__(kBlock) void k_spmv_sell_half(int N, const int *__restrict__ ia,
                                                           const int *__restrict__ off, const int *__restrict__ col,
                                                           const _Float16 *__restrict__ val,
                                                           const float *__restrict__ vsc, const TX *__restrict__ x,
                                                           TY *__restrict__ y, const double *__restrict__ bsub) {
    const int i = xcd_block() * kBlock + threadIdx.x;
    if (i >= N) return;
    const int l = i & 63;
    const int len = ia[i + 1] - ia[i];
    size_t p = (size_t)off[i >> 6] + l;
    TY s[5];
#pragma unroll
    for (int r = 0; r < 5; r++) s[r] = TY(0.0);
    for (int k = 0; k < len; k++, p += 64) {
        const TX *xj = x + 5 * (size_t)col[p];
        float xv[5];
#pragma unroll
        for (int c = 0; c < 5; c++) xv[c] = (float)xj[c];
        const _Float16 *A = val + 25 * (p - l) + l;
        const float sc = ld_stream(vsc + p);
#pragma unroll
        for (int r = 0; r < 5; r++) {
            float t = 0.0f;
#pragma unroll
            for (int c = 0; c < 5; c++) t += (float)ld_stream(A + 64 * (5 * r + c)) * xv[c];
            s[r] += (TY)(sc * t);
        }
    }
#pragma unroll
    for (int r = 0; r < 5; r++) {
        TY v = s[r];
        if (bsub) v = (TY)bsub[5 * (size_t)i + r] - v;
        y[5 * (size_t)i + r] = v;
    }
}

// ---------------------------------------------------------------------------
// Reference sweeps (MATH/src/MC_Iterative_Jacobi.c): Gauss-Seidel sweeps in one
// launch as a pipeline, LU-SGS one launch a half sweep
// ---------------------------------------------------------------------------
// No-pivot LU of the diagonal blocks, MC_Iterative_Jacobi.c:381-396
__global__ __launch_bounds__(kBlock) void k_gs_lu(int N, const int *iau, const double *a, double *lu) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= N) return;
    double L[25];
    for (int q = 0; q < 25; q++) L[q] = a[25 * (size_t)iau[r] + q];
    for (int k = 0; k < 4; k++) {
        for (int j = k + 1; j < 5; j++) L[5 * j + k] = L[5 * j + k] / L[5 * k + k];
        for (int j = k + 1; j < 5; j++)
            for (int i = k + 1; i < 5; i++) L[5 * i + j] -= L[5 * i + k] * L[5 * k + j];
    }
    for (int q = 0; q < 25; q++) lu[25 * (size_t)r + q] = L[q];
}

// A row's 5x5 block, of which its lane r holds row r, to all its lanes; sh as
// in FlowBlocks::dots.
__device__ __forceinline__ const double *flow_lu(double *sh, int r, const double *lr) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 5; q++) sh[5 * r + q] = lr[q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return sh;
}

// Forward Gauss-Seidel sweeps 0..S-1 in one launch (row update:
// MC_Iterative_Jacobi.c:410-450), rows handed over as in k_arnoldi_flow: sweep s
// writes its own version ver[s] of x, so row i of sweep s needs only its
// lower neighbours of sweep s and its upper ones (and itself) of sweep s - 1,
// and sweep s follows `reach` + 1 chunks behind sweep s - 1 instead of waiting
// for its end (reach: how many chunks ahead an upper neighbour can be,
// ensure_gs_schedule).  Items (chunk c, sweep s) go in ascending
// c + s (reach + 1), then s, so each needs only earlier ones.  The chain is about
// levels + 8 S rows long instead of levels * S: 20 sweeps of the 48x16x16 mesh
// (205 levels) took 64.3 ms with a launch per level, 1.39 ms so.
// x0: x before the first sweep.  rowrms[s][i]: row i's sum of sweep s.
__global__ __launch_bounds__(kBlock, 2) void k_gs_flow(int N, int nchunk, int reach, int S, const int *__restrict__ slots,
                                                    const int *__restrict__ ia, const int *__restrict__ ja,
                                                    const int *__restrict__ iau, const double *__restrict__ a,
                                                    const double *__restrict__ b, const double *__restrict__ lu,
                                                    const double *x0, double *ver, double *rowrms, int *flag) {
    const int lane = threadIdx.x & 63, slot = lane / 5, r = lane - 5 * slot, base = lane - r;
    __shared__ __align__(16) FlowLds<double> lds;
    double *sh = lds.v[threadIdx.x >> 6] + slot * FlowLds<double>::slot;
    // step t holds the items (t - s lag, s), lo <= s <= hi; first: the number of items before it
    const int lag = reach + 1, items = nchunk * S;
    int t = 0, first = 0, lo = 0, hi = 0;
    int *const ticket = flag + kFlagTicket;
    for (int w = flow_ticket(ticket); w < items; w = flow_ticket(ticket)) {
        while (w - first > hi - lo) {
            first += hi - lo + 1;
            t++;
            if (hi + 1 < S && t >= (hi + 1) * lag) hi++;
            if (t >= nchunk + lo * lag) lo++;
        }
        const int s = lo + w - first, c = t - s * lag;
        const int i = slot < 12 ? slots[12 * c + slot] : -1;
        const double *prev = s ? ver + (size_t)(s - 1) * 5 * N : x0;
        double *cur = ver + (size_t)s * 5 * N;
        const size_t ri = 5 * (size_t)(i >= 0 ? i : 0) + r;
        const int diag = i >= 0 ? iau[i] : 0;
        double rhs = 0.0, own = 0.0, lr[5] = {};
        if (i >= 0) {
            const int ke = ia[i + 1];
            rhs = b[ri];
            // the diagonal and upper blocks' products first: their values are
            // of the sweep before and mostly there; subtracted in block order
#pragma unroll
            for (int q = 0; q < 5; q++) lr[q] = lu[5 * ri + q];
            FlowBlocks<8, double, double> g;
            double tu[8], t[8];
            g.load(diag, ke, r, ja, a, prev);
            g.wait(flag);
            g.dots(sh, r, tu);
            own = tu[0];
            for (int k0 = ia[i]; k0 < diag; k0 += 8) {
                g.load(k0, diag, r, ja, a, cur);
                g.wait(flag);
                g.dots(sh, r, t);
#pragma unroll
                for (int u = 0; u < 8; u++) rhs -= t[u];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) rhs -= tu[u];
            for (int k0 = diag + 8; k0 < ke; k0 += 8) {
                g.load(k0, ke, r, ja, a, prev);
                g.wait(flag);
                g.dots(sh, r, t);
#pragma unroll
                for (int u = 0; u < 8; u++) rhs -= t[u];
            }
        }
        double sq = 0.0;
#pragma unroll
        for (int q = 0; q < 5; q++) {
            const double e = __shfl(rhs, base + q, 64);
            sq += e * e;
        }
        if (i >= 0 && r == 0) rowrms[(size_t)s * N + i] = sq;
        rhs += own;
        // every lane of the row solves with the LU factors of the diagonal block
        const double *L = flow_lu(sh, r, lr);
        double tv[5], xn[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
            tv[q] = __shfl(rhs, base + q, 64);
#pragma unroll
            for (int p = 0; p < q; p++) tv[q] -= L[5 * q + p] * tv[p];
        }
#pragma unroll
        for (int q = 4; q >= 0; q--) {
            xn[q] = tv[q];
#pragma unroll
            for (int p = 4; p > q; p--) xn[q] -= L[5 * q + p] * xn[p];
            xn[q] = xn[q] / L[5 * q + q];
        }
        double xr = xn[0];
#pragma unroll
        for (int q = 1; q < 5; q++) xr = r == q ? xn[q] : xr;
        if (i >= 0) flow_store(cur + ri, xr);
    }
}

// Pivoted LU of the diagonal blocks for the LU-SGS sweeps (the same factors
// in every sweep), MATH/src/LinearAlgebra.c:20-41: rows in pivot order, the
// order itself as five decimal digits.
__global__ __launch_bounds__(kBlock) void k_lusgs_lu(int N, const int *iau, const double *a, double *lu, int *piv) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= N) return;
    double A[5][5];
    int P[5];
    for (int i = 0; i < 5; i++)
        for (int j = 0; j < 5; j++) A[i][j] = a[25 * (size_t)iau[r] + 5 * i + j];
    for (int i = 0; i < 5; i++) P[i] = i;
    for (int c = 0; c < 5; c++) {
        double pm = A[P[c]][c];
        int pi = c;
        for (int i = c + 1; i < 5; i++)
            if (fabs(A[P[i]][c]) > fabs(pm)) {
                pm = A[P[i]][c];
                pi = i;
            }
        if (pi != c) {
            int tt = P[c];
            P[c] = P[pi];
            P[pi] = tt;
        }
        for (int i = c + 1; i < 5; i++) A[P[i]][c] /= A[P[c]][c];
        for (int i = c + 1; i < 5; i++)
            for (int j = c + 1; j < 5; j++) A[P[i]][j] -= A[P[i]][c] * A[P[c]][j];
    }
    int code = 0;
    for (int i = 4; i >= 0; i--) code = 10 * code + P[i];
    piv[r] = code;
    for (int i = 0; i < 5; i++)
        for (int j = 0; j < 5; j++) lu[25 * (size_t)r + 5 * i + j] = A[P[i]][j];
}

// One LU-SGS half sweep (row update: MC_Iterative_Jacobi.c:586-678,
// MATH/src/LinearAlgebra.c:117-155) in one launch, rows handed over as in
// k_arnoldi_flow: the neighbours swept before row i are read from cur, the others
// from prev, the result of the half sweep before.  next is left unset for the
// half sweep after this one.  Half sweeps run in opposite directions, so they
// do not overlap.
__global__ __launch_bounds__(kBlock, 2) void k_lusgs_flow(int nslots, const int *__restrict__ slots,
                                                       const int *__restrict__ ia, const int *__restrict__ ja,
                                                       const int *__restrict__ iau, const double *__restrict__ a,
                                                       const double *__restrict__ b, const double *__restrict__ lu,
                                                       const int *__restrict__ piv, const double *prev, double *cur,
                                                       double *next, int backward, int *flag, int *ticket,
                                                       int *next_ticket) {
    const int lane = threadIdx.x & 63, slot = lane / 5, r = lane - 5 * slot, base = lane - r;
    __shared__ __align__(16) FlowLds<double> lds;
    double *sh = lds.v[threadIdx.x >> 6] + slot * FlowLds<double>::slot;
    const int total = (nslots + 11) / 12;
    for (int w = flow_ticket(ticket); w < total; w = flow_ticket(ticket)) {
        if (w == 0 && lane == 0) st_coh(next_ticket, 0);
        const int t = 12 * w + slot;
        const int i = slot < 12 && t < nslots ? slots[t] : -1;
        const size_t ri = 5 * (size_t)(i >= 0 ? i : 0) + r;
        const int diag = i >= 0 ? iau[i] : 0;
        int code = 0;
        double rhs = 0.0, lr[5] = {};
        if (i >= 0) {
#pragma unroll
            for (int q = 0; q < 5; q++) lr[q] = lu[5 * ri + q];
            const int ke = ia[i + 1];
            code = piv[i];
            rhs = b[ri];
            flow_unset(next + ri);
            for (int side = 0; side < 2; side++) {
                const double *x = side == backward ? cur : prev;
                const int kb = side ? diag + 1 : ia[i], kn = side ? ke : diag;
                for (int k0 = kb; k0 < kn; k0 += 8) {
                    FlowBlocks<8, double, double> g;
                    double t[8];
                    g.load(k0, kn, r, ja, a, x);
                    g.wait(flag);
                    g.dots(sh, r, t);
#pragma unroll
                    for (int u = 0; u < 8; u++) rhs -= t[u];
                }
            }
        }
        const double *L = flow_lu(sh, r, lr);
        double y[5], xs[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
            y[q] = __shfl(rhs, base + code % 10, 64);
            code /= 10;
#pragma unroll
            for (int p = 0; p < q; p++) y[q] -= y[p] * L[5 * q + p];
        }
#pragma unroll
        for (int q = 4; q >= 0; q--) {
            xs[q] = y[q];
#pragma unroll
            for (int p = 4; p > q; p--) xs[q] -= xs[p] * L[5 * q + p];
            xs[q] /= L[5 * q + q];
        }
        double xr = xs[0];
#pragma unroll
        for (int q = 1; q < 5; q++) xr = r == q ? xs[q] : xr;
        if (i >= 0) flow_store(cur + ri, xr);
    }
}

__global__ __launch_bounds__(kBlock) void k_lusgs_init(int N, const double *b, double *x) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= N) return;
    double s = 0.0;
    for (int j = 0; j < 5; j++) s += b[5 * (size_t)r + j];
    s /= 5;
    for (int j = 0; j < 5; j++) flow_store(x + 5 * (size_t)r + j, s);  // read as handover words
}

// ---------------------------------------------------------------------------
// Krylov vector kernels (deterministic reductions)
// ---------------------------------------------------------------------------
// Sum over the wavefront, in every lane: the butterfly 32, 16, 8, 4, 2, 1.  Its
// last four steps stay within rows of 16 lanes whose values repeat with the
// step's period, so a rotation brings each lane its partner's value without
// the LDS crossbar.
template <int N>
__device__ __forceinline__ double row_ror(double v) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + N, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + N, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v += __shfl_xor(v, 32, 64);
    v += __shfl_xor(v, 16, 64);
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    return v;
}

// wave_sum of four values at once: the steps 32 and 16 exchange halves of two
// values' lanes, so that one addition serves both and the four sums end in one
// register, in the rows of 16 lanes: value 0 in row 0, 2 in 1, 1 in 2, 3 in 3.
__device__ __forceinline__ double swap_add32(double a, double b) {
    const long long x = __builtin_bit_cast(long long, a), y = __builtin_bit_cast(long long, b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]) +
           __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b) {
    const long long x = __builtin_bit_cast(long long, a), y = __builtin_bit_cast(long long, b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]) +
           __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
__device__ __forceinline__ double wave_sum4(double v0, double v1, double v2, double v3) {
    double v = swap_add16(swap_add32(v0, v1), swap_add32(v2, v3));
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    return v;
}

// Gram-Schmidt passes over the entries o + i0, o + i0 + stride, ... < o + n of a
// thread, in that order:
//   kDots        acc[k] += V_ki w_i
//   kUpdateDots  w_i -= h_k V_ki for k ascending (as CGS in the oracle), rounded
//                once to TV and stored; then acc[k] += V_ki w_i
//   kUpdateNorm  the same update; then acc[0] += w_i w_i
// U entries go together, so that their loads overlap: a thread takes one round
// trip to memory for U of its entries.
// kUpdateDots keeps the entries' V values in registers between the update and
// the products: a grid has at most kDotParts blocks, two wavefronts per SIMD,
// so registers are free (rereading them from the caches took 166 us at 24
// vectors of 4.08M FP32 entries, this 130 us with the final sums).  More than 41
// values of FP64 do not fit beside their sums: there V is read again, two
// entries at a time (gs_hold; steps 42 to 64 of the 192x64x64 mesh took 2.50 ms
// each with values spilled, 2.34 so).
enum GsMode { kDots, kUpdateDots, kUpdateNorm };

template <class TV, int NVMAX, GsMode M>
constexpr bool gs_hold = M == kUpdateDots && (sizeof(TV) == 4 || NVMAX <= 41);

template <class TV, int NVMAX, GsMode M, int U>
__device__ __forceinline__ void gs_entries(size_t o, size_t i, size_t stride, int nv, const TV *__restrict__ V,
                                           size_t ld, const double *__restrict__ h, TV *__restrict__ w, double *acc) {
    constexpr int NC = (NVMAX + 7) / 8;
    constexpr bool HOLD = gs_hold<TV, NVMAX, M>;
    double wi[U];
    TV vv[U][HOLD ? NVMAX : 8];
#pragma unroll
    for (int u = 0; u < U; u++) wi[u] = (double)w[o + i + u * stride];
    auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 8 * c; k < 8 * c + 8 && k < NVMAX; k++)
                if (k < nv) vv[u][HOLD ? k : k - 8 * c] = V[ld * k + o + i + u * stride];
    };
    auto dots = [&](int c) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 8 * c; k < 8 * c + 8 && k < NVMAX; k++)
                if (k < nv) acc[k] += (double)vv[u][HOLD ? k : k - 8 * c] * wi[u];
    };
#pragma unroll
    for (int c = 0; c < NC; c++) {
        if (8 * c >= nv) continue;
        load(c);
        if (HOLD) continue;
        if (M == kDots) {
            dots(c);
            continue;
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 8 * c; k < 8 * c + 8 && k < NVMAX; k++)
                if (k < nv) wi[u] = wi[u] - h[k] * (double)vv[u][k - 8 * c];
    }
    if (M == kDots) return;
    if (HOLD) {
#pragma unroll
        for (int k = 0; k < NVMAX; k++)
            if (k < nv) {
                const double hk = h[k];
#pragma unroll
                for (int u = 0; u < U; u++) wi[u] = wi[u] - hk * (double)vv[u][HOLD ? k : 0];
            }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const TV wt = (TV)wi[u];
        w[o + i + u * stride] = wt;
        wi[u] = (double)wt;
        if (M == kUpdateNorm) acc[0] += wi[u] * wi[u];
    }
    if (M == kUpdateNorm) return;
    if (HOLD) {
        // (the empty asm: an FP32 value is converted again rather than kept in
        // FP64 from the update on, which would double its registers)
        if (sizeof(TV) == 4) {
#pragma unroll
            for (int k = 0; k < NVMAX; k++)
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (k < nv) asm volatile("" : "+v"(vv[u][HOLD ? k : 0]));
        }
    } else {
        asm volatile("" ::: "memory");  // V is read again rather than kept
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
        if (8 * c >= nv) continue;
        if (!HOLD) load(c);
        dots(c);
    }
}

// Where the sums of one partition (a mesh, or a case of a union) go.
struct GsSums {
    double *words;  // [nd][P] partial sums of its P blocks, handed over as in k_arnoldi_flow; unset between launches
    double *out;    // [nd]
    double *host;   // [nd] the same in pinned host memory
};

// Block b of the P of a partition: the pass over its entries, then its partial
// sums (a butterfly within each wavefront, the four wavefront sums in order)
// into the words of dot k, and in the wavefronts of the last blocks the final
// sums: lane l adds partials l, l + 64, ... in order, then the butterfly.  These
// kGsTail blocks wait for the others, which wait for nothing, so a launch ends
// on any GPU that holds more than kGsTail blocks of every launch under way.  (A launch of its
// own for the final sums took 4-5 us, three times per Arnoldi step, and a copy
// of the sums to the host 3 us.)
constexpr int kGsTail = 8;
template <class TV, int NVMAX, GsMode M, int U>
__device__ __forceinline__ void gs_block(size_t o, int b, int P, size_t n, int nv, const TV *__restrict__ V, size_t ld,
                                         const double *__restrict__ h, TV *__restrict__ w, const GsSums &g,
                                         int *flag) {
    constexpr int NA = M == kUpdateNorm ? 1 : NVMAX;
    __shared__ double wsum[NA][kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t stride = (size_t)P * kBlock;
    double acc[NA];
#pragma unroll
    for (int k = 0; k < NA; k++) acc[k] = 0.0;
    size_t i = b * (size_t)kBlock + threadIdx.x;
    if (U > 1)
        for (; i + (U - 1) * stride < n; i += U * stride)
            gs_entries<TV, NVMAX, M, U>(o, i, stride, nv, V, ld, h, w, acc);
    for (; i < n; i += stride) gs_entries<TV, NVMAX, M, 1>(o, i, stride, nv, V, ld, h, w, acc);
    const int nd = M == kUpdateNorm ? 1 : nv;
    if (NA == 1) {
        const double v = wave_sum(acc[0]);
        if (lane == 0) wsum[0][wave] = v;
    } else {
        const int row = lane >> 4, at = row == 1 ? 2 : row == 2 ? 1 : row;
#pragma unroll
        for (int k = 0; k < NA; k += 4)
            if (k < nd) {
                const double v = wave_sum4(acc[k], k + 1 < NA ? acc[k + 1 < NA ? k + 1 : 0] : 0.0,
                                           k + 2 < NA ? acc[k + 2 < NA ? k + 2 : 0] : 0.0,
                                           k + 3 < NA ? acc[k + 3 < NA ? k + 3 : 0] : 0.0);
                if ((lane & 15) == 0 && k + at < nd) wsum[k + at][wave] = v;
            }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < nd; k += kBlock)
        flow_store(g.words + (size_t)k * P + b, ((wsum[k][0] + wsum[k][1]) + wsum[k][2]) + wsum[k][3]);
    const int tail = min(P, kGsTail);
    if (b < P - tail) return;
    for (int k = (P - 1 - b) * (kBlock / 64) + wave; k < nd; k += tail * (kBlock / 64)) {
        double *p = g.words + (size_t)k * P;
        double s = 0.0;
        for (int q = lane; q < P; q += 64 * 8) {
            unsigned long long v[8];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (q + 64 * u < P) v[u] = flow_load(p + q + 64 * u);
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (q + 64 * u < P) {
                    s += flow_wait(p + q + 64 * u, v[u], flag);
                    flow_unset(p + q + 64 * u);
                }
        }
        s = wave_sum(s);
        if (lane == 0) {
            g.out[k] = s;
            g.host[k] = s;
        }
    }
}

template <class TV, int NVMAX, GsMode M, int U>
__global__ __launch_bounds__(kBlock, 2) void k_gs(size_t n, int nv, const TV *__restrict__ V, size_t ld,
                                               const double *__restrict__ h, TV *__restrict__ w, GsSums g, int *flag) {
    gs_block<TV, NVMAX, M, U>(0, blockIdx.x, gridDim.x, n, nv, V, ld, h, w, g, flag);
}

// The same over a union of cases: block (c, b) of the segment map takes case
// c's range with its coefficients h[c] and leaves the sums in out[c] (rows of
// kBOut).  Blocks of a case are consecutive, and its last ones add up
// its partials, so however many cases there are, they wait for few.
template <class TV, int NVMAX, GsMode M>
__global__ __launch_bounds__(kBlock, 2) void k_gs_seg(const int2 *__restrict__ blk, const int *__restrict__ first,
                                                      const int *__restrict__ off, const int *__restrict__ len, int nv,
                                                      const TV *__restrict__ V, size_t ld,
                                                      const double *__restrict__ h, double *out, double *host,
                                                      TV *__restrict__ w, double *words, int *flag) {
    const int2 cb = blk[blockIdx.x];
    const int f = first[cb.x], P = first[cb.x + 1] - f;
    const size_t oc = (size_t)cb.x * kBOut;
    const GsSums g{words + (size_t)f * (kMaxKrylov + 1), out + oc, host + oc};
    gs_block<TV, NVMAX, M, 1>((size_t)off[cb.x], cb.y, P, (size_t)len[cb.x], nv, V, ld, h + oc, w, g, flag);
}

// Final sums of k_vsum_partial: dot k (block k) adds partials as gs_block does.
__global__ __launch_bounds__(64) void k_mdot_final(int nparts, int nv, const double *part, double *out) {
    const int k = blockIdx.x;
    double s = 0.0;
    for (int p = threadIdx.x; p < nparts; p += 64) s += part[(size_t)p * (kMaxKrylov + 1) + k];
    s = wave_sum(s);
    if (threadIdx.x == 0) out[k] = s;
}

// dst = src * (1/scale) with scale read from the device (scale = out[idx])
template <class TS, class TD>
__global__ __launch_bounds__(kBlock) void k_scale(size_t n, const TS *src, TD *dst, double denom) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        dst[i] = (TD)((double)src[i] / denom);
}

// dst = src / sqrt(*norm2): the Arnoldi normalisation with the norm read from
// device memory (the host evaluates the same correctly rounded sqrt for its
// Givens rotations), so the step can be enqueued without a host round trip.
template <class TS, class TD>
__global__ __launch_bounds__(kBlock) void k_scale_dev(size_t n, const TS *src, TD *dst, const double *norm2) {
    const double denom = sqrt(norm2[0]);
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        dst[i] = (TD)((double)src[i] / denom);
}

// x += sum_k y_k Z_k
template <class TV>
__global__ __launch_bounds__(kBlock) void k_xupdate(size_t n, int nv, const TV *__restrict__ Z, size_t ld,
                                                    const double *__restrict__ y, double *__restrict__ x) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
        double xi = x[i];
        for (int k = 0; k < nv; k++) xi = xi + y[k] * (double)Z[ld * k + i];
        x[i] = xi;
    }
}

// Partial sums of blockIdx.y vectors of n values, vector k into column k of
// the partials.
__global__ __launch_bounds__(kBlock) void k_vsum_partial(size_t n, const double *v, double *part) {
    __shared__ double sh[kBlock];
    v += (size_t)blockIdx.y * n;
    double acc = 0.0;
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) acc += v[i];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)blockIdx.x * (kMaxKrylov + 1) + blockIdx.y] = sh[0];
}

__global__ void k_fill(size_t n, double v, double *x) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) x[i] = v;
}

// ---- union of independent cases (batched solves) ------------------------
// dst = src / sqrt(out[c][slot]) (Arnoldi normalisation, per case)
template <class TS, class TD>
__global__ __launch_bounds__(kBlock) void k_scale_dev_seg(size_t n, const int *__restrict__ ecase, const TS *src,
                                                          TD *dst, const double *__restrict__ out, int slot) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
        const double denom = sqrt(out[(size_t)ecase[i / 5] * kBOut + slot]);
        dst[i] = (TD)((double)src[i] / denom);
    }
}

// dst = src / den[c] (first Krylov vector, per case)
template <class TS, class TD>
__global__ __launch_bounds__(kBlock) void k_scale_seg(size_t n, const int *__restrict__ ecase, const TS *src, TD *dst,
                                                      const double *__restrict__ den) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        dst[i] = (TD)((double)src[i] / den[(size_t)ecase[i / 5] * (kMaxKrylov + 1)]);
}

// x += sum_{k < kdim_c} y_{c,k} Z_k
template <class TV>
__global__ __launch_bounds__(kBlock) void k_xupdate_seg(size_t n, const int *__restrict__ ecase,
                                                        const TV *__restrict__ Z, size_t ld,
                                                        const double *__restrict__ y, const int *__restrict__ kdim,
                                                        double *__restrict__ x) {
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
        const int c = ecase[i / 5];
        const double *yc = y + (size_t)c * (kMaxKrylov + 1);
        double xi = x[i];
        for (int k = 0; k < kdim[c]; k++) xi = xi + yc[k] * (double)Z[ld * k + i];
        x[i] = xi;
    }
}

int grid_cap(size_t n, int cap) {
    size_t g = (n + kBlock - 1) / kBlock;
    if (g < 1) g = 1;
    return (int)(g < (size_t)cap ? g : cap);
}

}  // namespace

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------
int launch_jacobian(cfd_mesh *m, const cfd_params *p, int rhs_mode, int mixed) {
    const int nb = xcd_grid((m->N + 127) / 128);
    if (mixed) {
        JacArgs<float> a{m->N, m->NT, m->order, m->inc_ptr, m->sptr, m->nbr, m->soff, m->iau, m->d.isx, m->d.isy,
                         m->d.isz, m->d.qa, m->d.vol, m->dt, m->d.res, m->af, m->b, p->gamma, p->entropy_fix,
                         rhs_mode};
        hipLaunchKernelGGL(k_jacobian<float>, dim3(nb), dim3(128), 0, m->stream, a);
    } else {
        JacArgs<double> a{m->N, m->NT, m->order, m->inc_ptr, m->sptr, m->nbr, m->soff, m->iau, m->d.isx, m->d.isy,
                          m->d.isz, m->d.qa, m->d.vol, m->dt, m->d.res, m->a, m->b, p->gamma, p->entropy_fix,
                          rhs_mode};
        hipLaunchKernelGGL(k_jacobian<double>, dim3(nb), dim3(128), 0, m->stream, a);
    }
    CFD_HIP(m, hipGetLastError());
    m->jac_valid = true;
    m->jac_mixed = mixed != 0;
    m->prec_valid = false;
    m->asell_valid = false;
    return CFD_OK;
}

int launch_jacobian_fd(cfd_mesh *m, const cfd_params *p, int method, int iter, int add_time, int rhs_mode,
                       int mixed) {
    int fdm = method;
    if (fdm == CFD_JAC_FD_ALTERNATE) fdm = (iter % 2 == 0) ? CFD_JAC_FD_FORWARD : CFD_JAC_FD_BACKWARD;
    FdArgs a{};
    a.N = m->N;
    a.NT = m->NT;
    a.order = m->order;
    a.ip = m->inc_ptr;
    a.sptr = m->sptr;
    a.nbr = m->nbr;
    a.soff = m->soff;
    a.iau = m->iau;
    a.isx = m->d.isx;
    a.isy = m->d.isy;
    a.isz = m->d.isz;
    a.qa = m->d.qa;
    a.qb = m->d.qb;
    a.vol = m->d.vol;
    a.dt = m->dt;
    a.res = m->d.res;
    a.btype = m->btype;
    a.bcase = m->bcase;
    a.case_inf = m->case_inf;
    a.a = mixed ? nullptr : m->a;
    a.af = mixed ? m->af : nullptr;
    a.b = m->b;
    a.g = p->gamma;
    a.frac = p->limiter_order == 2 ? 0.5 : 0.0;
    a.coeff = fdm == CFD_JAC_FD_CENTRAL ? 0.5 : 1.0;
    a.efix = p->entropy_fix;
    a.rhs_mode = rhs_mode;
    a.add_time = add_time;
    a.order2 = p->order == 2;
    a.lim = p->limiter != CFD_LIM_NONE;
    a.plus = fdm == CFD_JAC_FD_CENTRAL || fdm == CFD_JAC_FD_FORWARD;
    a.minus = fdm == CFD_JAC_FD_CENTRAL || fdm == CFD_JAC_FD_BACKWARD;
    a.iter = iter;
    a.zpg = p->zpg_iter;
    a.free = BcFree<double>{p->inf_rho, p->inf_u, p->inf_v, p->inf_w, p->inf_p, p->outflow_p};
    a.flag = m->flag;
    const int nb = (int)((10 * (size_t)m->N + 127) / 128);
    if (p->flux == CFD_FLUX_HLLC)
        hipLaunchKernelGGL(k_jacobian_fd<CFD_FLUX_HLLC>, dim3(nb), dim3(128), 0, m->stream, a);
    else if (p->flux == CFD_FLUX_AUSMP)
        hipLaunchKernelGGL(k_jacobian_fd<CFD_FLUX_AUSMP>, dim3(nb), dim3(128), 0, m->stream, a);
    else
        hipLaunchKernelGGL(k_jacobian_fd<CFD_FLUX_ROE>, dim3(nb), dim3(128), 0, m->stream, a);
    CFD_HIP(m, hipGetLastError());
    m->jac_valid = true;
    m->jac_mixed = mixed != 0;
    m->prec_valid = false;
    m->asell_valid = false;
    return CFD_OK;
}

namespace {

// Block-SELL value arrays by storage type.
template <class TM>
struct SellVals;
template <>
struct SellVals<double> {
    static double *&a(cfd_mesh *m) { return m->asv; }
    static double *&l(cfd_mesh *m) { return m->lsv; }
    static double *&u(cfd_mesh *m) { return m->usv; }
    static double *&d(cfd_mesh *m) { return m->dsv; }
};
template <>
struct SellVals<float> {
    static float *&a(cfd_mesh *m) { return m->asvf; }
    static float *&l(cfd_mesh *m) { return m->lsvf; }
    static float *&u(cfd_mesh *m) { return m->usvf; }
    static float *&d(cfd_mesh *m) { return m->dsvf; }
};
// The BSR Jacobian by storage type.
template <class TM>
const TM *bsr_a(cfd_mesh *m);
template <>
const double *bsr_a<double>(cfd_mesh *m) { return m->a; }
template <>
const float *bsr_a<float>(cfd_mesh *m) { return m->af; }

// ILU(0) factors of A's blocks (in the pattern's order through src), a launch
// per level.
template <class TM>
void ilu0_levels(cfd_mesh *m, const LevelSchedule &ls, const int *ia, const int *ja, const int *iau, const int *src,
                 const TM *a, TM *lu, TM *dinv) {
    const int narrow = !m->ilu_long ? kIluNarrowRows : sizeof(TM) == 4 ? INT_MAX : kIluLongRows;
    for (int l = 0; l < ls.nlevels; l++) {
        const int b0 = ls.ptr[l], nr = ls.ptr[l + 1] - b0;
#define CFD_ILU(KERNEL, GRID, BLOCK)                                                                              \
    hipLaunchKernelGGL(KERNEL, dim3(GRID), dim3(BLOCK), 0, m->stream, nr, ls.rows + b0, ia, ja, iau, src, a, lu, \
                       dinv, (const TM *)lu, (const TM *)dinv, m->flag)
#define CFD_ILU_LEVEL(G)                                                                               \
    do {                                                                                               \
        const int rows = 4 * (12 / G);                                                                 \
        if (m->ilu_row > kIluSets<G> * G) CFD_ILU((k_ilu0_level<TM, G, true>), (nr + rows - 1) / rows, kBlock); \
        else CFD_ILU((k_ilu0_level<TM, G, false>), (nr + rows - 1) / rows, kBlock);                    \
    } while (0)
        if (nr <= narrow) CFD_ILU_LEVEL(12);
        else if (nr <= kIluFewRows) CFD_ILU_LEVEL(4);
        else if (m->ilu_row > kIluKeep) CFD_ILU((k_ilu0_rows<TM, true>), (nr + 11) / 12, 64);
        else CFD_ILU((k_ilu0_rows<TM, false>), (nr + 11) / 12, 64);
#undef CFD_ILU_LEVEL
#undef CFD_ILU
    }
}

template <class TM>
int build_prec(cfd_mesh *m, int kind, const TM *a, TM *lu, TM *dinv, bool half) {
    if (kind == CFD_PREC_ILU0_MC) {
        ilu0_levels(m, m->mc_lower, m->mc_ia, m->mc_ja, m->mc_iau, m->mc_src, a, lu, dinv);
        // block-SELL copies for the sweeps, FP16 with mixed = 2
        if constexpr (std::is_same<TM, float>::value) {
            if (half) {
                hipLaunchKernelGGL(k_to_sell_half, dim3(grid_cap((size_t)m->mcl_sell.nblk, 8192)), dim3(kBlock), 0,
                                   m->stream, (size_t)m->mcl_sell.nblk, m->mcl_sell.src, lu, m->lsvh, m->lsvs);
                hipLaunchKernelGGL(k_to_sell_half, dim3(grid_cap((size_t)m->mcu_sell.nblk, 8192)), dim3(kBlock), 0,
                                   m->stream, (size_t)m->mcu_sell.nblk, m->mcu_sell.src, lu, m->usvh, m->usvs);
                hipLaunchKernelGGL(k_to_sell_half, dim3(grid_cap((size_t)m->N, 8192)), dim3(kBlock), 0, m->stream,
                                   (size_t)m->N, nullptr, dinv, m->dsvh, m->dsvs);
            }
        }
        if (m->use_sell && !half) {
            hipLaunchKernelGGL(k_to_sell<TM>, dim3(grid_cap((size_t)m->mcl_sell.nblk, 8192)), dim3(kBlock), 0, m->stream,
                               (size_t)m->mcl_sell.nblk, m->mcl_sell.src, lu, SellVals<TM>::l(m));
            hipLaunchKernelGGL(k_to_sell<TM>, dim3(grid_cap((size_t)m->mcu_sell.nblk, 8192)), dim3(kBlock), 0, m->stream,
                               (size_t)m->mcu_sell.nblk, m->mcu_sell.src, lu, SellVals<TM>::u(m));
            hipLaunchKernelGGL(k_to_sell<TM>, dim3(grid_cap((size_t)m->N, 8192)), dim3(kBlock), 0, m->stream,
                               (size_t)m->N, nullptr, dinv, SellVals<TM>::d(m));
        }
    } else if (kind == CFD_PREC_ILU0) {
        ilu0_levels(m, m->lower, m->ia, m->ja, m->iau, nullptr, a, lu, dinv);
    } else if (kind == CFD_PREC_BJACOBI) {
        hipLaunchKernelGGL((k_block_inv<TM, TM>), dim3((m->N + kBlock - 1) / kBlock), dim3(kBlock), 0, m->stream,
                           m->N, m->iau, a, dinv, m->flag);
    }
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

// y = A x, or y = bsub - A x, with the block-SELL copy of the Jacobian.
template <class TM, class TX, class TY>
void spmv(cfd_mesh *m, const TX *x, TY *y, const double *bsub) {
    if (std::is_same<TM, float>::value && m->use_sell && m->asell_half)
        hipLaunchKernelGGL((k_spmv_sell_half<TX, TY>), dim3(xcd_grid((m->N + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                           m->stream, m->N, m->ia, m->a_sell.off, m->a_sell.col, m->asvh, m->asvs, x, y, bsub);
    else if (m->use_sell)
        hipLaunchKernelGGL((k_spmv_sell<TM, TX, TY>), dim3(xcd_grid((m->N + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                           m->stream,
                           m->N, m->ia, m->a_sell.off, m->a_sell.col, (const TM *)SellVals<TM>::a(m), x, y, bsub);
    else
        hipLaunchKernelGGL((k_spmv<TM, TX, TY>), dim3((int)((5 * (size_t)m->N + kBlock - 1) / kBlock)), dim3(kBlock),
                           0, m->stream, m->N, m->ia, m->ja, bsr_a<TM>(m), x, y, bsub);
}

// Whether the sweeps of this preconditioner run in one launch: in the natural
// order (hundreds of levels), and in the multicolour order on the BSR arrays,
// which meshes below kSellMinRows use.  20 Arnoldi steps with a launch per
// colour and in one launch, ms in FP64 and FP32: 63,504 rows 5.0 and 3.9, 3.5
// and 2.7; 104,448 rows 6.6 and 5.5, 5.1 and 4.2; 126,175 rows 7.1 and 6.2, 5.5
// and 4.9; Delaunay mesh of 100,000 11.2 and 9.0, 9.3 and 7.5.
bool flow_sweeps(const cfd_mesh *m, int kind) {
    return m->sync_free && (kind == CFD_PREC_ILU0 || (kind == CFD_PREC_ILU0_MC && !m->use_sell));
}

template <class TV>
TV *mc_work(cfd_mesh *m);
template <>
double *mc_work<double>(cfd_mesh *m) { return m->zp; }
template <>
float *mc_work<float>(cfd_mesh *m) { return m->zpf; }

template <class TM, class TV>
void apply_prec(cfd_mesh *m, int kind, const TM *lu, const TM *dinv, const TV *r, TV *z) {
    const size_t L = 5 * (size_t)m->N;
    if (kind == CFD_PREC_ILU0_MC && !m->use_sell) {
        TV *wk = mc_work<TV>(m);
        for (int pass = 0; pass < 2; pass++) {
            const LevelSchedule &ls = pass ? m->mc_upper : m->mc_lower;
            for (int l = 0; l < ls.nlevels; l++) {
                const int b0 = ls.ptr[l], nr = ls.ptr[l + 1] - b0;
                const int nwaves = (nr + 11) / 12;
                hipLaunchKernelGGL((k_trsv_mc<TM, TV>), dim3((nwaves + 3) / 4), dim3(kBlock), 0, m->stream, nr,
                                   ls.rows + b0, m->mc_ia, m->mc_ja, m->mc_iau, m->mc_perm, lu, dinv, r, wk, z, pass);
            }
        }
    } else if (kind == CFD_PREC_ILU0_MC && m->prec_half) {
        if constexpr (std::is_same<TM, float>::value && std::is_same<TV, float>::value) {
            float *wk = mc_work<float>(m);
            for (int pass = 0; pass < 2; pass++) {
                const BlockSell &bs = pass ? m->mcu_sell : m->mcl_sell;
                const _Float16 *val = pass ? m->usvh : m->lsvh;
                const float *vsc = pass ? m->usvs : m->lsvs;
                for (int t = 0; t < m->ncolor; t++) {
                    const int c = pass ? m->ncolor - 1 - t : t;
                    const int r0 = m->mc_cstart[c], r1 = m->mc_cstart[c + 1];
                    const int g = xcd_grid((r1 - (r0 & ~63) + kBlock - 1) / kBlock);
                    hipLaunchKernelGGL(k_trsv_mc_sell_half, dim3(g), dim3(kBlock), 0, m->stream, r0, r1, m->mc_ia,
                                       m->mc_iau, m->mc_perm, bs.off, bs.col, val, vsc, m->dsvh, m->dsvs, r, wk, z,
                                       pass);
                }
            }
        }
    } else if (kind == CFD_PREC_ILU0_MC) {
        // one launch per colour: forward in colour order, backward in reverse
        TV *wk = mc_work<TV>(m);
        const TM *dv = SellVals<TM>::d(m);
        for (int pass = 0; pass < 2; pass++) {
            const BlockSell &bs = pass ? m->mcu_sell : m->mcl_sell;
            const TM *val = pass ? SellVals<TM>::u(m) : SellVals<TM>::l(m);
            for (int t = 0; t < m->ncolor; t++) {
                const int c = pass ? m->ncolor - 1 - t : t;
                const int r0 = m->mc_cstart[c], r1 = m->mc_cstart[c + 1];
                const int g = xcd_grid((r1 - (r0 & ~63) + kBlock - 1) / kBlock);
                hipLaunchKernelGGL((k_trsv_mc_sell<TM, TV>), dim3(g), dim3(kBlock), 0, m->stream, r0, r1, m->mc_ia,
                                   m->mc_iau, m->mc_perm, bs.off, bs.col, val, dv, r, wk, z, pass);
            }
        }
    } else if (kind == CFD_PREC_ILU0) {
        for (int pass = 0; pass < 2; pass++) {
            const LevelSchedule &ls = pass ? m->upper : m->lower;
            for (int l = 0; l < ls.nlevels; l++) {
                const int b0 = ls.ptr[l], nr = ls.ptr[l + 1] - b0;
                const int nwaves = (nr + 11) / 12;
                hipLaunchKernelGGL((k_trsv_level<TM, TV>), dim3((nwaves + 3) / 4), dim3(kBlock), 0, m->stream, nr,
                                   ls.rows + b0, m->ia, m->ja, m->iau, lu, dinv, r, z, pass);
            }
        }
    } else if (kind == CFD_PREC_BJACOBI) {
        hipLaunchKernelGGL((k_bjac_apply<TM, TV>), dim3((int)((L + kBlock - 1) / kBlock)), dim3(kBlock), 0, m->stream,
                           m->N, dinv, r, z);
    } else {
        hipMemcpyAsync(z, r, sizeof(TV) * L, hipMemcpyDeviceToDevice, m->stream);
    }
}

// Entries that a thread of k_gs takes together: as many as registers hold
// where each walks four strides or more, else one.
template <class TV, int NVMAX>
constexpr int gs_unroll(GsMode M) {
    if (M != kUpdateDots || NVMAX == 8) return 4;
    if (sizeof(TV) == 4) return NVMAX <= 32 ? 4 : NVMAX <= 41 ? 2 : 1;
    return NVMAX <= 16 || NVMAX > 41 ? 2 : 1;
}

// One Gram-Schmidt pass of w against V_0..V_{nv-1} (coefficients at m->redout +
// hoff); sums to m->redout + off and m->hred + off.
template <class TV, GsMode M>
void gs_pass(cfd_mesh *m, int nv, const TV *V, size_t ld, int hoff, TV *w, int off) {
    const size_t L = 5 * (size_t)m->N;
    const int np = dot_parts(L);
    const double *h = m->redout + hoff;
    const GsSums g{m->red, m->redout + off, m->hred + off};
    const bool deep = L >= 4 * (size_t)np * kBlock;
    // NVMAX: the fewest unrolled vectors that cover nv
#define CFD_GS(NVMAX)                                                                                               \
    do {                                                                                                            \
        if (deep)                                                                                                   \
            hipLaunchKernelGGL((k_gs<TV, NVMAX, M, gs_unroll<TV, NVMAX>(M)>), dim3(np), dim3(kBlock), 0,            \
                               m->stream, L, nv, V, ld, h, w, g, m->flag);                                          \
        else                                                                                                        \
            hipLaunchKernelGGL((k_gs<TV, NVMAX, M, 1>), dim3(np), dim3(kBlock), 0, m->stream, L, nv, V, ld,  \
                               h, w, g, m->flag);                                                                   \
    } while (0)
    if (nv <= 8) CFD_GS(8);
    else if (nv <= 16) CFD_GS(16);
    else if (nv <= 32) CFD_GS(32);
    else if (nv <= 41) CFD_GS(41);
    else CFD_GS(kMaxKrylov + 1);
#undef CFD_GS
}

// The two sets of handover words of k_arnoldi_flow in the sweeps' work vector;
// step j of a cycle uses set j % 2 and leaves the other unset.
constexpr size_t kFlowWords = 3;  // vectors of a set

// Krylov basis of one storage type for restart length mk.  Each precision
// keeps its own basis, so alternating FP64 and mixed solves on one mesh
// allocates each once; a basis too short for a larger mk is replaced (the
// old one freed, after the stream is idle and the graphs captured on it are
// dropped), so the mesh's footprint never grows past one basis per
// precision.
int ensure_krylov(cfd_mesh *m, int mk, int precond, bool mixed) {
    const size_t L = 5 * (size_t)m->N;
    // the sweeps' work vector: two sets of handover words where they run in one
    // launch, else the permuted vector
    const int want = flow_sweeps(m, precond) ? 2 * (int)kFlowWords : 1;
    int &nzp = mixed ? m->nzp32 : m->nzp64;
    if (nzp < want) {
        if (nzp) {
            CFD_HIP(m, hipStreamSynchronize(m->stream));
            drop_krylov_graphs(m);
        }
        nzp = 0;
        if (mixed) {
            cfd_dfree(m, m->zpf);
            m->zpf = (float *)cfd_dalloc(m, sizeof(float) * want * L);
        } else {
            cfd_dfree(m, m->zp);
            m->zp = (double *)cfd_dalloc(m, sizeof(double) * want * L);
        }
        if (mixed ? !m->zpf : !m->zp)
            return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (work vector of the sweeps)");
        nzp = want;
    }
    if (!m->r) m->r = (double *)cfd_dalloc(m, sizeof(double) * L);
    if (!m->r) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (Krylov)");
    int &have = mixed ? m->kry_m32 : m->kry_m64;
    if (have >= mk) return CFD_OK;
    if (have > 0) {
        CFD_HIP(m, hipStreamSynchronize(m->stream));
        drop_krylov_graphs(m);
    }
    if (mixed) {
        cfd_dfree(m, m->Vf);
        cfd_dfree(m, m->Zf);
        cfd_dfree(m, m->wf);
        m->Vf = (float *)cfd_dalloc(m, sizeof(float) * L * (mk + 1));
        m->Zf = (float *)cfd_dalloc(m, sizeof(float) * L * mk);
        m->wf = (float *)cfd_dalloc(m, sizeof(float) * L);
        have = 0;
        if (!m->Vf || !m->Zf || !m->wf) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (Krylov FP32)");
    } else {
        cfd_dfree(m, m->V);
        cfd_dfree(m, m->Z);
        cfd_dfree(m, m->w);
        m->V = (double *)cfd_dalloc(m, sizeof(double) * L * (mk + 1));
        m->Z = (double *)cfd_dalloc(m, sizeof(double) * L * mk);
        m->w = (double *)cfd_dalloc(m, sizeof(double) * L);
        have = 0;
        if (!m->V || !m->Z || !m->w) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (Krylov)");
    }
    have = mk;
    return CFD_OK;
}

// Steps 1-3 of arnoldi_step in one launch: V_j (from w, where norm2 is given),
// Z_j and, on the BSR arrays, w = A Z_j; returns whether w was formed.
template <class TM, class TV>
bool flow_step(cfd_mesh *m, const TM *a, const TM *lu, const TM *dinv, TV *vj, TV *zj, TV *w, int j,
               const double *norm2) {
    const size_t L = 5 * (size_t)m->N;
    const bool mc = m->prec_kind == CFD_PREC_ILU0_MC;
    const LevelSchedule &lo = mc ? m->mc_lower : m->lower, &up = mc ? m->mc_upper : m->upper;
    TV *set = mc_work<TV>(m);
    FlowStep<TM, TV> f{};
    f.nf = lo.n12;
    f.nb = up.n12;
    f.np = m->use_sell ? 0 : m->N;
    f.sf = lo.slots12;
    f.sb = up.slots12;
    f.ia = mc ? m->mc_ia : m->ia;
    f.ja = mc ? m->mc_ja : m->ja;
    f.iau = mc ? m->mc_iau : m->iau;
    f.perm = mc ? m->mc_perm : nullptr;
    f.lu = lu;
    f.dinv = dinv;
    f.w = w;
    f.norm2 = norm2;
    f.v = vj;
    f.z = zj;
    f.y = w;
    f.aia = m->ia;
    f.aja = m->ja;
    f.a = a;
    f.words = set + (j & 1) * kFlowWords * L;
    f.other = set + (1 - (j & 1)) * kFlowWords * L;
    f.L = L;
    f.flag = m->flag;
    f.ticket = m->flag + kFlagTicket + (j & 1);
    f.next_ticket = m->flag + kFlagTicket + 1 - (j & 1);
    const int chunks = (f.nf + 11) / 12 + (f.nb + 11) / 12 + (f.np + 11) / 12;
    const int64_t width = m->N / 12 / std::max(1, std::max(lo.nlevels, up.nlevels));
    hipLaunchKernelGGL((k_arnoldi_flow<TM, TV>), dim3(flow_blocks(m, chunks, width)), dim3(kBlock), 0, m->stream, f);
    return f.np > 0;
}

// Unsets the first set of handover words, before step 0 of a cycle.
template <class TV>
void flow_begin(cfd_mesh *m) {
    const size_t n = kFlowWords * 5 * (size_t)m->N;
    hipLaunchKernelGGL(k_flow_unset<TV>, dim3(grid_cap(n, 4096)), dim3(kBlock), 0, m->stream, n, mc_work<TV>(m),
                       m->flag + kFlagTicket);
}

// One Arnoldi step j of FGMRES: V_j = w / ||w|| (j > 0, norm of the previous
// step), Z_j = M^-1 V_j, w = A Z_j, two CGS passes against V_0..V_j and
// ||w||^2, whose sums the passes leave on the host too.  The sequence depends
// only on j and the mesh's buffers, so it is captured once per j as a graph.
template <class TM, class TV>
void arnoldi_step(cfd_mesh *m, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z, TV *w, int j) {
    const size_t L = 5 * (size_t)m->N;
    const int gN = grid_cap(L, 4096);
    TV *vj = V + L * j, *zj = Z + L * j;
    const double *norm2 = j > 0 ? m->redout + 2 * (kMaxKrylov + 1) : nullptr;
    bool product = false;
    if (flow_sweeps(m, m->prec_kind)) {
        product = flow_step<TM, TV>(m, a, lu, dinv, vj, zj, w, j, norm2);
    } else {
        if (norm2) hipLaunchKernelGGL((k_scale_dev<TV, TV>), dim3(gN), dim3(kBlock), 0, m->stream, L, w, vj, norm2);
        apply_prec<TM, TV>(m, m->prec_kind, lu, dinv, vj, zj);
    }
    if (!product) spmv<TM, TV, TV>(m, zj, w, nullptr);
    // CGS2: h1 = V^T w, w -= V h1, h2 = V^T w, w -= V h2, ||w||^2 (each
    // update fused with the reduction after it)
    gs_pass<TV, kDots>(m, j + 1, V, L, 0, w, 0);
    gs_pass<TV, kUpdateDots>(m, j + 1, V, L, 0, w, kMaxKrylov + 1);
    gs_pass<TV, kUpdateNorm>(m, j + 1, V, L, kMaxKrylov + 1, w, 2 * (kMaxKrylov + 1));
}

// Enqueues Arnoldi step j, replaying its captured graph (captured on first use).
template <class TM, class TV>
int enqueue_step(cfd_mesh *m, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z, TV *w, int j, int mk) {
    if (!m->use_graphs) {
        arnoldi_step<TM, TV>(m, a, lu, dinv, V, Z, w, j);
        CFD_HIP(m, hipGetLastError());
        return CFD_OK;
    }
    KrylovGraphs &kg = m->kgraph;
    if (kg.key != (const void *)V || kg.prec != m->prec_kind || kg.m != mk || kg.lu != (const void *)lu) {
        drop_krylov_graphs(m);
        kg.key = V;
        kg.lu = lu;
        kg.prec = m->prec_kind;
        kg.m = mk;
        kg.exec.assign(mk, nullptr);
    }
    if (!kg.exec[j]) {
        // Relaxed mode: other threads driving other meshes may call
        // allocation or synchronous copy functions meanwhile.  If the capture
        // still fails, this mesh falls back to direct launches of the same
        // sequence.
        hipGraph_t g = nullptr;
        hipGraphExec_t ex = nullptr;
        hipError_t e;
        {
            std::unique_lock<std::shared_mutex> lk(cfd_capture_mutex());
            e = hipStreamBeginCapture(m->stream, hipStreamCaptureModeRelaxed);
            if (e == hipSuccess) {
                arnoldi_step<TM, TV>(m, a, lu, dinv, V, Z, w, j);
                e = hipStreamEndCapture(m->stream, &g);
            }
            if (e == hipSuccess) e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
            if (g) hipGraphDestroy(g);
        }
        if (e != hipSuccess || !ex) {
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(m->stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
                hipGraph_t g2 = nullptr;
                (void)hipStreamEndCapture(m->stream, &g2);
                if (g2) hipGraphDestroy(g2);
            }
            (void)hipGetLastError();
            m->use_graphs = false;
            drop_krylov_graphs(m);
            arnoldi_step<TM, TV>(m, a, lu, dinv, V, Z, w, j);
            CFD_HIP(m, hipGetLastError());
            return CFD_OK;
        }
        kg.exec[j] = ex;
    }
    CFD_HIP(m, hipGraphLaunch((hipGraphExec_t)kg.exec[j], m->stream));
    return CFD_OK;
}

// The same per case of a union: coefficients at m->bred[c][hslot..], sums to
// m->bred[c][slot..] and m->hbred[c][slot..].
template <class TV, GsMode M>
void gs_pass_seg(cfd_mesh *m, int nv, const TV *V, size_t ld, int hslot, TV *w, int slot) {
    const SegMap &sg = m->seg_dot;
#define CFD_GS_SEG(NVMAX)                                                                                            \
    hipLaunchKernelGGL((k_gs_seg<TV, NVMAX, M>), dim3(sg.nblocks), dim3(kBlock), 0, m->stream, sg.blk, sg.first,     \
                       sg.off, sg.len, nv, V, ld, m->bred + hslot, m->bred + slot, m->hbred + slot, w, m->bpart, m->flag)
    if (nv <= 8) CFD_GS_SEG(8);
    else if (nv <= 16) CFD_GS_SEG(16);
    else if (nv <= 32) CFD_GS_SEG(32);
    else if (nv <= 41) CFD_GS_SEG(41);
    else CFD_GS_SEG(kMaxKrylov + 1);
#undef CFD_GS_SEG
}

// Arnoldi step j of the batched FGMRES: the operations of arnoldi_step with
// per-case dots, coefficients and norms.
template <class TM, class TV>
void arnoldi_step_batch(cfd_mesh *m, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z, TV *w, int j) {
    const size_t L = 5 * (size_t)m->N;
    const int gN = grid_cap(L, 4096);
    TV *vj = V + L * j, *zj = Z + L * j;
    if (j > 0)
        hipLaunchKernelGGL((k_scale_dev_seg<TV, TV>), dim3(gN), dim3(kBlock), 0, m->stream, L, m->ecase, w, vj,
                           m->bred, 2 * (kMaxKrylov + 1));
    bool product = false;
    if (flow_sweeps(m, m->prec_kind)) product = flow_step<TM, TV>(m, a, lu, dinv, vj, zj, w, j, nullptr);
    else apply_prec<TM, TV>(m, m->prec_kind, lu, dinv, vj, zj);
    if (!product) spmv<TM, TV, TV>(m, zj, w, nullptr);
    gs_pass_seg<TV, kDots>(m, j + 1, V, L, 0, w, 0);
    gs_pass_seg<TV, kUpdateDots>(m, j + 1, V, L, 0, w, kMaxKrylov + 1);
    gs_pass_seg<TV, kUpdateNorm>(m, j + 1, V, L, kMaxKrylov + 1, w, 2 * (kMaxKrylov + 1));
}

template <class TM, class TV>
int enqueue_step_batch(cfd_mesh *m, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z, TV *w, int j, int mk) {
    if (!m->use_graphs) {
        arnoldi_step_batch<TM, TV>(m, a, lu, dinv, V, Z, w, j);
        CFD_HIP(m, hipGetLastError());
        return CFD_OK;
    }
    KrylovGraphs &kg = m->kgraph_b;
    if (kg.key != (const void *)V || kg.prec != m->prec_kind || kg.m != mk || kg.lu != (const void *)lu) {
        CfdRuntimeGuard guard;
        for (auto &g : kg.exec)
            if (g) hipGraphExecDestroy((hipGraphExec_t)g);
        kg.key = V;
        kg.lu = lu;
        kg.prec = m->prec_kind;
        kg.m = mk;
        kg.exec.assign(mk, nullptr);
    }
    if (!kg.exec[j]) {
        // Relaxed mode: other threads driving other meshes may call
        // allocation or synchronous copy functions meanwhile.  If the capture
        // still fails, this mesh falls back to direct launches of the same
        // sequence.
        hipGraph_t g = nullptr;
        hipGraphExec_t ex = nullptr;
        hipError_t e;
        {
            std::unique_lock<std::shared_mutex> lk(cfd_capture_mutex());
            e = hipStreamBeginCapture(m->stream, hipStreamCaptureModeRelaxed);
            if (e == hipSuccess) {
                arnoldi_step_batch<TM, TV>(m, a, lu, dinv, V, Z, w, j);
                e = hipStreamEndCapture(m->stream, &g);
            }
            if (e == hipSuccess) e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
            if (g) hipGraphDestroy(g);
        }
        if (e != hipSuccess || !ex) {
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(m->stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
                hipGraph_t g2 = nullptr;
                (void)hipStreamEndCapture(m->stream, &g2);
                if (g2) hipGraphDestroy(g2);
            }
            (void)hipGetLastError();
            m->use_graphs = false;
            drop_krylov_graphs(m);
            arnoldi_step_batch<TM, TV>(m, a, lu, dinv, V, Z, w, j);
            CFD_HIP(m, hipGetLastError());
            return CFD_OK;
        }
        kg.exec[j] = ex;
    }
    CFD_HIP(m, hipGraphLaunch((hipGraphExec_t)kg.exec[j], m->stream));
    return CFD_OK;
}

// The solve's error flags to m->hflag; an error if a single-launch sweep gave up
// a wait.
int sweep_gave_up(cfd_mesh *m) {
    m->hflag[2] = m->hflag[3] = 0;
    CFD_HIP(m, hipMemcpyAsync(m->hflag, m->flag, 4 * sizeof(int), hipMemcpyDeviceToHost, m->stream));
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    return m->hflag[3] ? cfd_set_error(m->ctx, CFD_E_HIP, "a single-launch sweep exceeded its wait bound") : CFD_OK;
}

// Batched restarted FGMRES(m): every case of the union runs the algorithm of
// fgmres() on its own rows, in lockstep; a case that has converged (or is
// not being solved) keeps riding along but its results are not used.
template <class TM, class TV>
int fgmres_batch(cfd_mesh *m, const cfd_linsolve_opts *o, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z,
                 TV *w, const std::vector<char> &solve, std::vector<int> &iters, std::vector<double> &fres,
                 std::vector<int> &status) {
    const int K = m->ncase, mk = o->krylov_m;
    const size_t L = 5 * (size_t)m->N;
    const int gN = grid_cap(L, 4096);
    const size_t ldc = kMaxKrylov + 1;
    hipLaunchKernelGGL(k_fill, dim3(gN), dim3(kBlock), 0, m->stream, L, 0.0, m->x);
    CFD_HIP(m, hipMemcpyAsync(m->r, m->b, sizeof(double) * L, hipMemcpyDeviceToDevice, m->stream));
    gs_pass_seg<double, kDots>(m, 1, m->r, 0, 0, m->r, 0);
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    std::vector<double> beta(K), tol(K), res(K);
    std::vector<char> live(K), cyc(K), step(K);
    std::vector<int> kdim(K);
    std::vector<double> H((size_t)K * (mk + 1) * mk, 0.0), cs((size_t)K * mk), sn((size_t)K * mk),
        gv((size_t)K * (mk + 1)), hcol(mk + 2), y((size_t)mk);
    iters.assign(K, 0);
    fres.assign(K, 0.0);
    status.assign(K, CFD_OK);
    for (int c = 0; c < K; c++) {
        beta[c] = sqrt(m->hbred[(size_t)c * kBOut]);
        tol[c] = o->rtol * beta[c];
        res[c] = beta[c];
        live[c] = solve[c] && beta[c] > tol[c] && beta[c] > 0.0;
    }
    for (int cycle = 0; cycle <= o->max_restarts; cycle++) {
        bool any = false;
        for (int c = 0; c < K; c++) {
            cyc[c] = step[c] = live[c];
            kdim[c] = 0;
            any = any || live[c];
            m->hbcoef[(size_t)c * ldc] = live[c] ? beta[c] : 1.0;
            for (int i = 0; i <= mk; i++) gv[(size_t)c * (mk + 1) + i] = 0.0;
            gv[(size_t)c * (mk + 1)] = beta[c];
        }
        if (!any) break;
        CFD_HIP(m, hipMemcpyAsync(m->bcoef, m->hbcoef, sizeof(double) * ldc * K, hipMemcpyHostToDevice, m->stream));
        hipLaunchKernelGGL((k_scale_seg<double, TV>), dim3(gN), dim3(kBlock), 0, m->stream, L, m->ecase, m->r, V,
                           m->bcoef);
        if (flow_sweeps(m, m->prec_kind)) flow_begin<TV>(m);
        for (int j = 0; j < mk; j++) {
            int rc = enqueue_step_batch<TM, TV>(m, a, lu, dinv, V, Z, w, j, mk);
            if (rc) return rc;
            CFD_HIP(m, hipStreamSynchronize(m->stream));
            bool stepping = false;
            for (int c = 0; c < K; c++) {
                if (!step[c]) continue;
                const double *hr = m->hbred + (size_t)c * kBOut;
                double *Hc = H.data() + (size_t)c * (mk + 1) * mk, *csc = cs.data() + (size_t)c * mk,
                       *snc = sn.data() + (size_t)c * mk, *gvc = gv.data() + (size_t)c * (mk + 1);
                for (int k = 0; k <= j; k++) hcol[k] = 0.0 + hr[k];
                for (int k = 0; k <= j; k++) hcol[k] += hr[kMaxKrylov + 1 + k];
                const double hn = sqrt(hr[2 * (kMaxKrylov + 1)]);
                hcol[j + 1] = hn;
                for (int k = 0; k < j; k++) {
                    const double t = csc[k] * hcol[k] + snc[k] * hcol[k + 1];
                    hcol[k + 1] = -snc[k] * hcol[k] + csc[k] * hcol[k + 1];
                    hcol[k] = t;
                }
                const double den = sqrt(hcol[j] * hcol[j] + hcol[j + 1] * hcol[j + 1]);
                csc[j] = hcol[j] / den;
                snc[j] = hcol[j + 1] / den;
                hcol[j] = den;
                hcol[j + 1] = 0.0;
                gvc[j + 1] = -snc[j] * gvc[j];
                gvc[j] = csc[j] * gvc[j];
                for (int k = 0; k <= j; k++) Hc[(size_t)k * mk + j] = hcol[k];
                iters[c]++;
                kdim[c] = j + 1;
                res[c] = fabs(gvc[j + 1]);
                if (!(res[c] == res[c])) {
                    rc = sweep_gave_up(m);
                    if (rc) return rc;
                    // this case fails on its own (as its solve alone would);
                    // its correction is dropped and the other cases go on
                    status[c] = CFD_E_NONFINITE;
                    step[c] = cyc[c] = live[c] = false;
                    continue;
                }
                if (res[c] <= tol[c] || hn == 0.0) step[c] = false;
                stepping = stepping || step[c];
            }
            if (!stepping) break;
        }
        for (int c = 0; c < K; c++) {
            double *yc = m->hbcoef + (size_t)c * ldc;
            for (int k = 0; k <= kMaxKrylov; k++) yc[k] = 0.0;
            m->hbkdim[c] = cyc[c] ? kdim[c] : 0;
            if (!cyc[c]) continue;
            const double *Hc = H.data() + (size_t)c * (mk + 1) * mk, *gvc = gv.data() + (size_t)c * (mk + 1);
            for (int k = kdim[c] - 1; k >= 0; k--) {
                double t = gvc[k];
                for (int q = k + 1; q < kdim[c]; q++) t -= Hc[(size_t)k * mk + q] * y[q];
                y[k] = t / Hc[(size_t)k * mk + k];
            }
            for (int k = 0; k < kdim[c]; k++) yc[k] = y[k];
        }
        CFD_HIP(m, hipMemcpyAsync(m->bcoef, m->hbcoef, sizeof(double) * ldc * K, hipMemcpyHostToDevice, m->stream));
        CFD_HIP(m, hipMemcpyAsync(m->bkdim, m->hbkdim, sizeof(int) * K, hipMemcpyHostToDevice, m->stream));
        hipLaunchKernelGGL(k_xupdate_seg<TV>, dim3(gN), dim3(kBlock), 0, m->stream, L, m->ecase, Z, L, m->bcoef,
                           m->bkdim, m->x);
        any = false;
        for (int c = 0; c < K; c++) {
            if (cyc[c] && res[c] <= tol[c]) live[c] = false;
            any = any || live[c];
        }
        if (!any) break;
        // true residual for the restart
        spmv<TM, double, double>(m, m->x, m->r, m->b);
        gs_pass_seg<double, kDots>(m, 1, m->r, 0, 0, m->r, 0);
        CFD_HIP(m, hipStreamSynchronize(m->stream));
        for (int c = 0; c < K; c++) {
            if (!live[c]) continue;
            beta[c] = sqrt(m->hbred[(size_t)c * kBOut]);
            res[c] = beta[c];
            live[c] = cycle < o->max_restarts && beta[c] > tol[c] && beta[c] > 0.0;
        }
    }
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    for (int c = 0; c < K; c++) fres[c] = res[c];
    return CFD_OK;
}

// Restarted right-preconditioned FGMRES(m) with CGS2; same algorithm as
// orc_fgmres.  TM: matrix and preconditioner storage, TV: Krylov vectors.
template <class TM, class TV>
int fgmres(cfd_mesh *m, const cfd_linsolve_opts *o, const TM *a, const TM *lu, const TM *dinv, TV *V, TV *Z, TV *w,
           cfd_linsolve_stats *st) {
    const int mk = o->krylov_m;
    const size_t L = 5 * (size_t)m->N;
    const int gN = grid_cap(L, 4096);
    double *hr = m->hred;
    // x0 = 0; r0 = b
    hipLaunchKernelGGL(k_fill, dim3(gN), dim3(kBlock), 0, m->stream, L, 0.0, m->x);
    CFD_HIP(m, hipMemcpyAsync(m->r, m->b, sizeof(double) * L, hipMemcpyDeviceToDevice, m->stream));
    gs_pass<double, kDots>(m, 1, m->r, 0, 0, m->r, 0);
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    const double bnorm = sqrt(hr[0]);
    const double tol = o->rtol * bnorm;
    double beta = bnorm, res = bnorm;
    std::vector<double> H((size_t)(mk + 1) * mk, 0.0), cs(mk), sn(mk), gv(mk + 1), hcol(mk + 2), y(mk);
    int total = 0, cycles = 0;
    st->b_norm = bnorm;
    for (int cycle = 0; cycle <= o->max_restarts && beta > tol && beta > 0.0; cycle++) {
        cycles++;
        hipLaunchKernelGGL((k_scale<double, TV>), dim3(gN), dim3(kBlock), 0, m->stream, L, m->r, V, beta);
        if (flow_sweeps(m, m->prec_kind)) flow_begin<TV>(m);
        for (int i = 0; i <= mk; i++) gv[i] = 0.0;
        gv[0] = beta;
        int kdim = 0;
        for (int j = 0; j < mk; j++) {
            int rc = enqueue_step<TM, TV>(m, a, lu, dinv, V, Z, w, j, mk);
            if (rc) return rc;
            CFD_HIP(m, hipStreamSynchronize(m->stream));
            for (int k = 0; k <= j; k++) hcol[k] = 0.0 + hr[k];
            for (int k = 0; k <= j; k++) hcol[k] += hr[kMaxKrylov + 1 + k];
            const double hn = sqrt(hr[2 * (kMaxKrylov + 1)]);
            hcol[j + 1] = hn;
            for (int k = 0; k < j; k++) {
                const double t = cs[k] * hcol[k] + sn[k] * hcol[k + 1];
                hcol[k + 1] = -sn[k] * hcol[k] + cs[k] * hcol[k + 1];
                hcol[k] = t;
            }
            const double den = sqrt(hcol[j] * hcol[j] + hcol[j + 1] * hcol[j + 1]);
            cs[j] = hcol[j] / den;
            sn[j] = hcol[j + 1] / den;
            hcol[j] = den;
            hcol[j + 1] = 0.0;
            gv[j + 1] = -sn[j] * gv[j];
            gv[j] = cs[j] * gv[j];
            for (int k = 0; k <= j; k++) H[(size_t)k * mk + j] = hcol[k];
            total++;
            kdim = j + 1;
            res = fabs(gv[j + 1]);
            if (!(res == res)) {
                // a wait that was given up leaves NaNs: that is the failure then
                rc = sweep_gave_up(m);
                return rc ? rc : cfd_set_error(m->ctx, CFD_E_NONFINITE, "FGMRES: non-finite residual");
            }
            // the next step starts with V_{j+1} = w / hn (k_scale_dev)
            if (res <= tol || hn == 0.0) break;
        }
        for (int k = kdim - 1; k >= 0; k--) {
            double s = gv[k];
            for (int t = k + 1; t < kdim; t++) s -= H[(size_t)k * mk + t] * y[t];
            y[k] = s / H[(size_t)k * mk + k];
        }
        for (int k = 0; k < kdim; k++) hr[k] = y[k];
        CFD_HIP(m, hipMemcpyAsync(m->redout + 3 * (kMaxKrylov + 1), hr, sizeof(double) * kdim, hipMemcpyHostToDevice,
                                  m->stream));
        hipLaunchKernelGGL(k_xupdate<TV>, dim3(gN), dim3(kBlock), 0, m->stream, L, kdim, Z, L,
                           m->redout + 3 * (kMaxKrylov + 1), m->x);
        if (res <= tol) break;
        // true residual for the restart
        spmv<TM, double, double>(m, m->x, m->r, m->b);
        gs_pass<double, kDots>(m, 1, m->r, 0, 0, m->r, 0);
        CFD_HIP(m, hipStreamSynchronize(m->stream));
        beta = sqrt(hr[0]);
        res = beta;
    }
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    st->iterations = total;
    st->restarts = cycles > 0 ? cycles - 1 : 0;
    st->final_res = res;
    return CFD_OK;
}

}  // namespace

namespace {
int prepare_fgmres(cfd_mesh *m, const cfd_linsolve_opts *o);
int read_solve_flags(cfd_mesh *m);
}  // namespace

void drop_krylov_graphs(cfd_mesh *m) {
    CfdRuntimeGuard guard;
    for (KrylovGraphs *kg : {&m->kgraph, &m->kgraph_b}) {
        for (auto &g : kg->exec)
            if (g) hipGraphExecDestroy((hipGraphExec_t)g);
        kg->exec.clear();
        kg->key = nullptr;
    }
}

// The schedule of k_gs_flow (host, on the mesh's first Gauss-Seidel solve).
// Row i of sweep s takes step p_i + lag s: p_i is above the p of every lower
// neighbour and at least p_k + 1 - lag for every upper neighbour k.  The levels
// do with a lag one above their largest jump from a row to an upper neighbour
// (50 on the bump channels of 200 levels).  A smaller lag is sought by raising
// p: three passes settle lag 8 on the channels, where 7 is the least there is.
// On unstructured meshes hardly any lag is below the jumps, and p rises without
// end: a lag is given up when p passes twice the levels.  (Lags tried in turn
// up to the levels, sixteen passes each, took 600 ms for 200,000 rows of a
// Delaunay mesh, this 40.)  reach: the largest number of chunks from a row to
// an upper neighbour.
static int ensure_gs_schedule(cfd_mesh *m) {
    if (m->gs.slots12) return CFD_OK;
    const int N = m->N, nl = m->lower.nlevels;
    std::vector<int> lev(N), p, chunk(N), s12, rows(N);
    CFD_HIP(m, cfd_memcpy(rows.data(), m->lower.rows, sizeof(int) * rows.size(), hipMemcpyDeviceToHost));
    for (int l = 0; l < nl; l++)
        for (int t = m->lower.ptr[l]; t < m->lower.ptr[l + 1]; t++) lev[rows[t]] = l;
    // largest of of(row, upper neighbour) over the pattern
    auto most_over_upper = [&](const std::vector<int> &of) {
        std::atomic<int> most{0};
        cfd_parallel_for(N, [&](int64_t i0, int64_t i1) {
            int d = 0;
            for (int i = (int)i0; i < (int)i1; i++)
                for (int k = m->h_iau[i] + 1; k < m->h_ia[i + 1]; k++) d = std::max(d, of[m->h_ja[k]] - of[i]);
            for (int v = most; d > v && !most.compare_exchange_weak(v, d);) {
            }
        });
        return most.load();
    };
    const int jump = most_over_upper(lev);
    bool settled = false;
    for (int lag = 8; lag <= jump && !settled; lag *= 4) {
        p = lev;
        bool raised = true, high = false;
        for (int pass = 0; pass < 8 && raised && !high; pass++) {
            raised = false;
            for (int i = 0; i < N && !high; i++) {
                int t = p[i];
                for (int k = m->h_ia[i]; k < m->h_iau[i]; k++) t = std::max(t, p[m->h_ja[k]] + 1);
                for (int k = m->h_iau[i] + 1; k < m->h_ia[i + 1]; k++) t = std::max(t, p[m->h_ja[k]] + 1 - lag);
                raised = raised || t > p[i];
                high = t > 2 * nl;
                p[i] = t;
            }
        }
        settled = !raised && !high;
    }
    if (!settled) p = lev;
    LevelSchedule &ls = m->gs;
    ls.nlevels = *std::max_element(p.begin(), p.end()) + 1;
    ls.ptr.assign(ls.nlevels + 1, 0);
    for (int i = 0; i < N; i++) ls.ptr[p[i] + 1]++;
    for (int l = 0; l < ls.nlevels; l++) ls.ptr[l + 1] += ls.ptr[l];
    std::vector<int> at(ls.ptr.begin(), ls.ptr.end() - 1);
    for (int i = 0; i < N; i++) rows[at[p[i]]++] = i;
    pad_levels(ls.ptr, rows, 12, s12);
    for (size_t t = 0; t < s12.size(); t++)
        if (s12[t] >= 0) chunk[s12[t]] = (int)(t / 12);
    m->gs_reach = most_over_upper(chunk);
    int *d = (int *)cfd_dalloc(m, sizeof(int) * s12.size());
    if (!d) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (sweep schedule)");
    CFD_HIP(m, cfd_memcpy(d, s12.data(), sizeof(int) * s12.size(), hipMemcpyHostToDevice));
    ls.slots12 = d;
    ls.n12 = (int)s12.size();
    return CFD_OK;
}

// Scratch of the Gauss-Seidel sweeps, all of it written before it is read.
struct GsScratch {
    double *lu;    // [N][25] LU factors of the diagonal blocks
    double *rows;  // [nver][N] per-row sums of the RMS of each sweep
    double *ver;   // [nver][N][5] x after each sweep
    int nver;      // sweeps per launch
};

// Forward block Gauss-Seidel sweeps of MC_Iterative_Block_LU_Jacobi_CRS
// (MATH/src/MC_Iterative_Jacobi.c:346-535), up to g.nver to a launch; the
// sweeps end with the first whose RMS is small enough, so x is its version.
// More than one sweep to a launch needs the schedule ls and reach of
// ensure_gs_schedule; one at a time runs on any lower level schedule.
static int gs_sweeps(cfd_mesh *m, int sweeps, const LevelSchedule &ls, int reach, const GsScratch &g,
                     cfd_linsolve_stats *st) {
    const size_t L = 5 * (size_t)m->N;
    hipLaunchKernelGGL(k_gs_lu, dim3((m->N + kBlock - 1) / kBlock), dim3(kBlock), 0, m->stream, m->N, m->iau, m->a,
                       g.lu);
    hipLaunchKernelGGL(k_fill, dim3(grid_cap(L, 4096)), dim3(kBlock), 0, m->stream, L, 0.0, m->x);
    const int nchunk = ls.n12 / 12, np = grid_cap(m->N, kDotParts);
    double rms = 0.0;
    int it = 0;
    for (bool done = false; it < sweeps && !done;) {
        const int S = std::min(g.nver, sweeps - it);
        // a step's chunks of every sweep under way; more than 256 workgroups lose
        // where sweeps hardly overlap (Delaunay meshes) and gain little elsewhere:
        // 1.53, 1.39, 1.54 ms at 128, 256 and 512 (48x16x16 mesh), 0.79, 0.82, 0.94
        // (24x8x8), 27.7, 21.3, 31.3 (Delaunay, 200,000 rows), 24.4, 16.1, 14.1
        // (192x64x64, ten sweeps)
        const int64_t under = std::min<int64_t>(S, nchunk / (reach + 1) + 1);
        const int64_t width = std::min<int64_t>(nchunk * under / ls.nlevels, 399);
        hipLaunchKernelGGL(k_flow_unset<double>, dim3(grid_cap(S * L, 4096)), dim3(kBlock), 0, m->stream, S * L, g.ver,
                           m->flag + kFlagTicket);
        hipLaunchKernelGGL(k_gs_flow, dim3(flow_blocks(m, (int64_t)nchunk * S, width)), dim3(kBlock), 0, m->stream, m->N, nchunk, reach, S, ls.slots12, m->ia, m->ja, m->iau, m->a, m->b, g.lu,
                           m->x, g.ver, g.rows, m->flag);
        // row RMS of each sweep: ordered reduction of the per-row sums
        hipLaunchKernelGGL(k_vsum_partial, dim3(np, S), dim3(kBlock), 0, m->stream, (size_t)m->N, g.rows, m->red);
        hipLaunchKernelGGL(k_mdot_final, dim3(S), dim3(64), 0, m->stream, np, S, m->red, m->redout);
        CFD_HIP(m, hipMemcpyAsync(m->hred, m->redout, sizeof(double) * S, hipMemcpyDeviceToHost, m->stream));
        const int rc = sweep_gave_up(m);
        if (rc) return rc;
        int last = S;
        for (int s = 0; s < S && !done; s++) {
            rms = sqrt(m->hred[s] / (double)m->N);
            done = rms < 100.0 * DBL_EPSILON;
            if (done) last = s + 1;
        }
        it += last;
        CFD_HIP(m, hipMemcpyAsync(m->x, g.ver + (size_t)(last - 1) * L, sizeof(double) * L, hipMemcpyDeviceToDevice,
                                  m->stream));
    }
    st->iterations = it;
    st->final_res = rms;
    return CFD_OK;
}

// Scratch of cfd_linsolve_gs_noalloc: the LU factors of the diagonal blocks
// (25 values per row), the per-row sums (1) and x after the sweep (5) of
// meshes of up to kNoAllocMaxNodes nodes, 8.1 MB.  Each GPU holds its own copy
// until the process ends; host code uses the address hipGetSymbolAddress
// returns for the current GPU (kept per context), never the array's name.
// Every call on a GPU shares that GPU's copy, so calls that overlap on one GPU
// race.
static __device__ __align__(256) double scratch[31 * (size_t)kNoAllocMaxNodes];

double *noalloc_scratch_address(hipError_t *err) {
    void *p = nullptr;
    *err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    return *err == hipSuccess ? (double *)p : nullptr;
}

int run_gs_noalloc(cfd_mesh *m, int sweeps, cfd_linsolve_stats *st) {
    *st = cfd_linsolve_stats{};
    if (!m->jac_valid) return cfd_set_error(m->ctx, CFD_E_STATE, "cfd_linsolve_gs_noalloc: no Jacobian assembled");
    if (m->jac_mixed) return cfd_set_error(m->ctx, CFD_E_ARG, "cfd_linsolve_gs_noalloc: needs an FP64 Jacobian");
    if (m->N > kNoAllocMaxNodes)
        return cfd_set_error(m->ctx, CFD_E_ARG,
                             "cfd_linsolve_gs_noalloc: %d nodes exceed the scratch array's %d (use cfd_linsolve)",
                             m->N, kNoAllocMaxNodes);
    if (!m->ctx->noalloc_scratch)
        return cfd_set_error(m->ctx, CFD_E_HIP, "cfd_linsolve_gs_noalloc: scratch array address unavailable");
    double *base = m->ctx->noalloc_scratch;
    const size_t n = kNoAllocMaxNodes;
    CFD_HIP(m, hipMemsetAsync(m->flag, 0, 4 * sizeof(int), m->stream));
    const GsScratch g{base, base + 25 * n, base + 26 * n, 1};
    const int rc = gs_sweeps(m, sweeps > 0 ? sweeps : 10000, m->lower, 0, g, st);
    if (rc) return rc;
    CFD_HIP(m, hipGetLastError());
    CFD_HIP(m, hipStreamSynchronize(m->stream));
    return CFD_OK;
}

// Gauss-Seidel sweeps per launch: each keeps a version of x (48 bytes per node
// with its row sums).  A further sweep in a launch costs reach + 1 chunks of
// the chain, a further launch the whole chain, so as many as fit 512 MB, 32 at
// most, and fewer where the device has less left: one will do.
static int gs_versions(const cfd_mesh *m, int sweeps) {
    const int64_t fit = (512LL << 20) / (48 * (int64_t)m->N);
    return (int)std::max<int64_t>(1, std::min<int64_t>({fit, 32, sweeps}));
}

// Room for `want` versions in m->gsver, at least `need`; how many there are.
static int ensure_gs_room(cfd_mesh *m, int want, int need) {
    if (m->gs_nver >= want) return want;
    if (m->gs_short && m->gs_nver >= need) return m->gs_nver;
    if (m->gs_nver) {
        CfdRuntimeGuard g;
        if (hipStreamSynchronize(m->stream) != hipSuccess) return 0;
    }
    cfd_dfree(m, m->gsver);
    m->gsver = nullptr;
    m->gs_nver = 0;
    for (int v = want; v >= need && !m->gsver; v = v > need ? std::max(need, v / 2) : 0) {
        m->gsver = (double *)cfd_dalloc(m, sizeof(double) * 6 * (size_t)m->N * v);
        if (m->gsver) m->gs_nver = v;
        else m->gs_short = true;
    }
    return m->gs_nver;
}

int run_linsolve(cfd_mesh *m, const cfd_linsolve_opts *o, cfd_linsolve_stats *st) {
    if (!m->jac_valid) return cfd_set_error(m->ctx, CFD_E_STATE, "cfd_linsolve: no Jacobian assembled");
    *st = cfd_linsolve_stats{};
    CFD_HIP(m, hipMemsetAsync(m->flag, 0, 4 * sizeof(int), m->stream));
    if (o->solver == CFD_SOLVER_BLOCK_GS || o->solver == CFD_SOLVER_LUSGS) {
        if (m->jac_mixed) return cfd_set_error(m->ctx, CFD_E_ARG, "reference sweeps need an FP64 Jacobian");
        const int sweeps = o->sweeps > 0 ? o->sweeps : (o->solver == CFD_SOLVER_BLOCK_GS ? 10000 : 100);
        const bool gs = o->solver == CFD_SOLVER_BLOCK_GS;
        if (!m->gslu) m->gslu = (double *)cfd_dalloc(m, sizeof(double) * 25 * (size_t)m->N);
        const int nver = m->gslu ? ensure_gs_room(m, gs ? gs_versions(m, sweeps) : 3, gs ? 1 : 3) : 0;
        if (!nver) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (sweeps)");
        const size_t L = 5 * (size_t)m->N;
        double *ver = m->gsver;  // [nver][N][5], then [nver][N] row sums (GS) or the pivot orders (LU-SGS)
        if (gs) {
            // one sweep to a launch where there is no room for more, or for their schedule
            int rc = nver > 1 ? ensure_gs_schedule(m) : CFD_OK;
            const bool one = nver == 1 || rc == CFD_E_OOM;
            if (rc && !one) return rc;
            rc = gs_sweeps(m, sweeps, one ? m->lower : m->gs, one ? 0 : m->gs_reach,
                           GsScratch{m->gslu, ver + L * nver, ver, one ? 1 : nver}, st);
            if (rc) return rc;
        } else {
            int *piv = (int *)(ver + 3 * L);
            hipLaunchKernelGGL(k_lusgs_init, dim3((m->N + kBlock - 1) / kBlock), dim3(kBlock), 0, m->stream, m->N,
                               m->b, m->x);
            hipLaunchKernelGGL(k_lusgs_lu, dim3((m->N + kBlock - 1) / kBlock), dim3(kBlock), 0, m->stream, m->N, m->iau,
                               m->a, m->gslu, piv);
            hipLaunchKernelGGL(k_flow_unset<double>, dim3(grid_cap(L, 4096)), dim3(kBlock), 0, m->stream, L, ver,
                               m->flag + kFlagTicket);
            // half sweep h writes version h % 3, reads h - 1 and clears h + 1
            for (int h = 0; h < 2 * sweeps; h++) {
                const LevelSchedule &ls = h % 2 ? m->upper : m->lower;
                hipLaunchKernelGGL(k_lusgs_flow, dim3(flow_blocks(m, ls.n12 / 12, m->N / 12 / ls.nlevels)),
                                   dim3(kBlock), 0, m->stream, ls.n12, ls.slots12, m->ia, m->ja, m->iau, m->a, m->b, m->gslu, piv,
                                   h ? ver + (h + 2) % 3 * L : m->x, ver + h % 3 * L, ver + (h + 1) % 3 * L, h % 2,
                                   m->flag, m->flag + kFlagTicket + h % 2, m->flag + kFlagTicket + 1 - h % 2);
            }
            CFD_HIP(m, hipMemcpyAsync(m->x, ver + (2 * sweeps - 1) % 3 * L, sizeof(double) * L,
                                      hipMemcpyDeviceToDevice, m->stream));
            CFD_HIP(m, hipGetLastError());
            st->iterations = sweeps;
            return read_solve_flags(m);
        }
        CFD_HIP(m, hipGetLastError());
        CFD_HIP(m, hipStreamSynchronize(m->stream));
        return CFD_OK;
    }
    int rc = prepare_fgmres(m, o);
    if (rc) return rc;
    if (o->mixed)
        rc = fgmres<float, float>(m, o, m->af, m->luf, m->dinvf, m->Vf, m->Zf, m->wf, st);
    else
        rc = fgmres<double, double>(m, o, m->a, m->lu, m->dinv, m->V, m->Z, m->w, st);
    if (rc) return rc;
    return read_solve_flags(m);
}

int run_linsolve_batch(cfd_mesh *m, const cfd_linsolve_opts *o, const std::vector<char> &solve,
                       std::vector<int> &iters, std::vector<double> &final_res, std::vector<int> &status) {
    if (m->ncase < 1) return cfd_set_error(m->ctx, CFD_E_STATE, "batched solve on a mesh that is not a union of cases");
    if (!m->jac_valid) return cfd_set_error(m->ctx, CFD_E_STATE, "batched linsolve: no Jacobian assembled");
    if (o->solver != CFD_SOLVER_FGMRES) return cfd_set_error(m->ctx, CFD_E_ARG, "batched solves use FGMRES");
    CFD_HIP(m, hipMemsetAsync(m->flag, 0, 4 * sizeof(int), m->stream));
    int rc = prepare_fgmres(m, o);
    if (rc) return rc;
    if (o->mixed)
        rc = fgmres_batch<float, float>(m, o, m->af, m->luf, m->dinvf, m->Vf, m->Zf, m->wf, solve, iters, final_res,
                                        status);
    else
        rc = fgmres_batch<double, double>(m, o, m->a, m->lu, m->dinv, m->V, m->Z, m->w, solve, iters, final_res,
                                          status);
    if (rc) return rc;
    return read_solve_flags(m);
}

namespace {

// Jacobian precision check, Krylov workspace and preconditioner for FGMRES.
// Allocates the block-SELL value arrays of storage type TM: A always, the
// multicolour factors for that preconditioner.
template <class TM>
int ensure_sell(cfd_mesh *m, int precond, bool half, bool half_a) {
    if (!m->use_sell) return CFD_OK;
    TM *&av = SellVals<TM>::a(m);
    if (!av) av = (TM *)cfd_dalloc(m, sizeof(TM) * 25 * (size_t)m->a_sell.nblk);
    if (!av) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (block-SELL Jacobian)");
    if (precond != CFD_PREC_ILU0_MC) return CFD_OK;
    if (half) {
        const size_t nl = std::max<int64_t>(m->mcl_sell.nblk, 64), nu = std::max<int64_t>(m->mcu_sell.nblk, 64),
                     nd = ((size_t)m->N + 63) / 64 * 64;
        if (half_a && !m->asvh) m->asvh = (_Float16 *)cfd_dalloc(m, sizeof(_Float16) * 25 * (size_t)m->a_sell.nblk);
        if (half_a && !m->asvs) m->asvs = (float *)cfd_dalloc(m, sizeof(float) * (size_t)m->a_sell.nblk);
        if (half_a && (!m->asvh || !m->asvs))
            return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (FP16 A)");
        if (!m->lsvh) m->lsvh = (_Float16 *)cfd_dalloc(m, sizeof(_Float16) * 25 * nl);
        if (!m->usvh) m->usvh = (_Float16 *)cfd_dalloc(m, sizeof(_Float16) * 25 * nu);
        if (!m->dsvh) m->dsvh = (_Float16 *)cfd_dalloc(m, sizeof(_Float16) * 25 * nd);
        if (!m->lsvs) m->lsvs = (float *)cfd_dalloc(m, sizeof(float) * nl);
        if (!m->usvs) m->usvs = (float *)cfd_dalloc(m, sizeof(float) * nu);
        if (!m->dsvs) m->dsvs = (float *)cfd_dalloc(m, sizeof(float) * nd);
        if (!m->lsvh || !m->usvh || !m->dsvh || !m->lsvs || !m->usvs || !m->dsvs)
            return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (FP16 block-SELL factors)");
        return CFD_OK;
    }
    TM *&lv = SellVals<TM>::l(m), *&uv = SellVals<TM>::u(m), *&dv = SellVals<TM>::d(m);
    if (!lv) lv = (TM *)cfd_dalloc(m, sizeof(TM) * 25 * (size_t)std::max<int64_t>(m->mcl_sell.nblk, 64));
    if (!uv) uv = (TM *)cfd_dalloc(m, sizeof(TM) * 25 * (size_t)std::max<int64_t>(m->mcu_sell.nblk, 64));
    if (!dv) dv = (TM *)cfd_dalloc(m, sizeof(TM) * 25 * (((size_t)m->N + 63) / 64 * 64));
    if (!lv || !uv || !dv) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (block-SELL factors)");
    return CFD_OK;
}

// The rows of a schedule in whole chunks of 12 (LevelSchedule::slots12), for
// schedules that do not hold them from the mesh's creation.
int ensure_slots12(cfd_mesh *m, LevelSchedule &ls) {
    if (ls.slots12) return CFD_OK;
    std::vector<int> rows(m->N), s12;
    CFD_HIP(m, cfd_memcpy(rows.data(), ls.rows, sizeof(int) * rows.size(), hipMemcpyDeviceToHost));
    pad_levels(ls.ptr, rows, 12, s12);
    int *d = (int *)cfd_dalloc(m, sizeof(int) * s12.size());
    if (!d) return cfd_set_error(m->ctx, CFD_E_OOM, "out of device memory (sweep schedule)");
    CFD_HIP(m, cfd_memcpy(d, s12.data(), sizeof(int) * s12.size(), hipMemcpyHostToDevice));
    ls.slots12 = d;
    ls.n12 = (int)s12.size();
    return CFD_OK;
}

int prepare_fgmres(cfd_mesh *m, const cfd_linsolve_opts *o) {
    if (o->krylov_m < 1 || o->krylov_m > kMaxKrylov)
        return cfd_set_error(m->ctx, CFD_E_ARG, "krylov_m must be in [1, %d]", kMaxKrylov);
    if (o->precond < CFD_PREC_NONE || o->precond > CFD_PREC_ILU0_MC)
        return cfd_set_error(m->ctx, CFD_E_ARG, "unknown preconditioner %d", o->precond);
    if (o->mixed < 0 || o->mixed > 3) return cfd_set_error(m->ctx, CFD_E_ARG, "mixed must be 0, 1, 2 or 3");
    const bool mixed = o->mixed != 0;
    // FP16 copies of the factors (mixed >= 2) and of A (mixed = 3), for the
    // multicolour ILU(0) on the block-SELL kernels
    const bool sell_mc = o->precond == CFD_PREC_ILU0_MC && m->use_sell;
    const bool half = o->mixed >= 2 && sell_mc, half_a = o->mixed == 3 && sell_mc;
    if (mixed != m->jac_mixed)
        return cfd_set_error(m->ctx, CFD_E_ARG, "Jacobian precision does not match linsolve precision");
    int rc = ensure_krylov(m, o->krylov_m, o->precond, mixed);
    if (rc) return rc;
    // the partial sums of the Gram-Schmidt passes (their buffers serve other
    // reductions between linear solves)
    const size_t nw = (size_t)(kMaxKrylov + 1) * (m->ncase ? m->seg_dot.nblocks : dot_parts(5 * (size_t)m->N));
    hipLaunchKernelGGL(k_flow_unset<double>, dim3(grid_cap(nw, 4096)), dim3(kBlock), 0, m->stream, nw,
                       m->ncase ? m->bpart : m->red, (int *)nullptr);
    if (o->precond == CFD_PREC_ILU0_MC && flow_sweeps(m, o->precond)) {
        rc = ensure_slots12(m, m->mc_lower);
        if (!rc) rc = ensure_slots12(m, m->mc_upper);
        if (rc) return rc;
    }
    rc = mixed ? ensure_sell<float>(m, o->precond, half, half_a)
               : ensure_sell<double>(m, o->precond, false, false);
    if (rc) return rc;
    if (m->use_sell && (!m->asell_valid || m->asell_half != half_a)) {
        if (m->asell_half != half_a) drop_krylov_graphs(m);  // captured steps launch the other SpMV kernel
        m->asell_half = half_a;
        if (half_a)
            hipLaunchKernelGGL(k_to_sell_half, dim3(grid_cap((size_t)m->a_sell.nblk, 8192)), dim3(kBlock), 0,
                               m->stream, (size_t)m->a_sell.nblk, m->a_sell.src, m->af, m->asvh, m->asvs);
        else if (mixed)
            hipLaunchKernelGGL(k_to_sell<float>, dim3(grid_cap((size_t)m->a_sell.nblk, 8192)), dim3(kBlock), 0,
                               m->stream, (size_t)m->a_sell.nblk, m->a_sell.src, m->af, m->asvf);
        else
            hipLaunchKernelGGL(k_to_sell<double>, dim3(grid_cap((size_t)m->a_sell.nblk, 8192)), dim3(kBlock), 0,
                               m->stream, (size_t)m->a_sell.nblk, m->a_sell.src, m->a, m->asv);
        CFD_HIP(m, hipGetLastError());
        m->asell_valid = true;
    }
    if (!m->prec_valid || m->prec_kind != o->precond || m->prec_mixed != mixed || m->prec_half != half) {
        if (m->prec_half != half) drop_krylov_graphs(m);  // captured steps launch the other sweep kernels
        m->prec_kind = o->precond;
        m->prec_mixed = mixed;
        m->prec_half = half;
        if (mixed) {
            if ((o->precond == CFD_PREC_ILU0 || o->precond == CFD_PREC_ILU0_MC) && !m->luf)
                m->luf = (float *)cfd_dalloc(m, sizeof(float) * 25 * (size_t)m->nnz);
            if (o->precond != CFD_PREC_NONE && !m->dinvf) m->dinvf = (float *)cfd_dalloc(m, sizeof(float) * 25 * (size_t)m->N);
            rc = build_prec<float>(m, o->precond, m->af, m->luf, m->dinvf, half);
        } else {
            if ((o->precond == CFD_PREC_ILU0 || o->precond == CFD_PREC_ILU0_MC) && !m->lu)
                m->lu = (double *)cfd_dalloc(m, sizeof(double) * 25 * (size_t)m->nnz);
            if (o->precond != CFD_PREC_NONE && !m->dinv) m->dinv = (double *)cfd_dalloc(m, sizeof(double) * 25 * (size_t)m->N);
            rc = build_prec<double>(m, o->precond, m->a, m->lu, m->dinv, false);
        }
        if (rc) return rc;
        m->prec_valid = true;
    }
    return CFD_OK;
}

// Error flags raised by the preconditioner and the sweeps.
int read_solve_flags(cfd_mesh *m) {
    const int rc = sweep_gave_up(m);
    if (m->hflag[2]) return cfd_set_error(m->ctx, CFD_E_SINGULAR, "zero pivot in %d diagonal blocks", m->hflag[2]);
    return rc;
}

}  // namespace
