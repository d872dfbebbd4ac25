// rk3w.hip -- the explicit Wray Runge-Kutta momentum predictor and the transposed steps of its
// checkpointed adjoint, on gfx950.  Compiled with FP contraction off: the forward stage update is
// the reference's VecCopy / VecAXPY sequence evaluated per element in the same order.
//
// Forward stage i (the low-storage scheme of UeqnRK3CN_W, src/solvers/ueqn_solvers.c:1508-1583,
// beta / delta of :1518-1520, the whole right-hand side explicit):
//   k_rk3w_update        Ucont = (Ucont + dt beta_i Rhs) + (-1.0 dt delta_i) Rhs_o into the owned
//                        range of the local ucont, and Rhs_o = Rhs (:1533-1541, :1563-1569)
// Adjoint (the transpose of each forward step, in reverse order; no reference counterpart):
//   k_rk3w_adj_combine   cotangent of the stage's Rhs from the two stage updates that read it
//   k_ghosts_adj         transpose of resetCellPeriodicFluxes' boundary copies (inline.h:5496-5514) and of the
//                        periodic ghost scatter (DMLocalToLocal)
//   k_c2c_adj_solve      transpose of contravariantToCartesian's 3x3 solve (src/ueqn.c:571-613)
//   k_c2c_adj_gather     transpose of its face averages (inline.h:4307-4310), added with FormU's ucont
//                        cotangent to the global one
//   k_face_resets_adj    transpose of resetFacePeriodicFluxesVector's face-0 copies (inline.h:5357-5451), then
//                        of resetNoPenetrationFluxes (inline.h:5262-5355): the zeroed fluxes carry no
//                        cotangent; a zeroGradient flux only where it was not clipped
#include "kernels.h"

namespace tosca {

namespace {

__device__ __forceinline__ long owned_local(const Geo &g, long q) {
    const int i = (int)(q % g.mx);
    const long r = q / g.mx;
    const int j = (int)(r % g.my), k = (int)(r / g.my);
    return g.L(k, j, i);
}

__device__ __forceinline__ long gidx(const Geo &g, int k, int j, int i) { return ((long)k * g.my + j) * g.mx + i; }

// one thread per owned double
__global__ void k_rk3w_update(double *ucont, const double *rhs, double *rhs_o, double a, double b, Geo g, long n) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    double *u = ucont + 3 * owned_local(g, t / 3) + t % 3;
    const double r = rhs[t];
    double v = *u;
    v = v + a * r;
    v = v + b * rhs_o[t];
    *u = v;
    rhs_o[t] = r;
}

// rbar = a xbar + carry (the cotangent of this stage's Rhs: from the next state, a = dt beta_i, and
// from the following stage's Rhs_o term, carry); carry = b xbar (b = -1.0 dt delta_i: the cotangent of
// the previous stage's Rhs through this stage's Rhs_o term)
__global__ void k_rk3w_adj_combine(const double *xbar, double *carry, double *rbar, double a, double b, long n) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double x = xbar[t];
    rbar[t] = a * x + carry[t];
    carry[t] = b * x;
}

// Transpose of resetCellPeriodicFluxes and the wraps, as a gather: a point of the interior range of the
// periodic axes collects the cotangents of its copies, the indices whose ghost_source it is (four on a
// wrapped axis of four points, the smallest); they keep theirs, which the transposed
// contravariantToCartesian does not read.  One thread per point next to the periodic boundaries, of three
// components.  Bound by the launch: 13 us at 128 x 96 x 64 with two periodic axes, where the six launches
// that scattered one axis and side at a time took 40.
__device__ __forceinline__ int copies(int x, int m, int per, int (&c)[5]) {
    int n = 0;
    c[n++] = x;
    if (per == TOSCA_PERIODIC_NONE) return n;
    const int w = per == TOSCA_PERIODIC_WRAP ? GW : 0;
    for (int y = -w; y <= 0; y++)
        if (ghost_source(y, m, per, RESET_CELL) == x) c[n++] = y;
    for (int y = m - 1; y < m + w; y++)
        if (ghost_source(y, m, per, RESET_CELL) == x) c[n++] = y;
    return n;
}
__global__ void __launch_bounds__(256) k_ghosts_adj(double *a, Geo g, Shell S) {
    int i, j, k, ci[5], cj[5], ck[5];
    if (!shell_point(S, blockIdx.x * blockDim.x + threadIdx.x, i, j, k)) return;
    const int ni = copies(i, g.mx, g.per[0], ci), nj = copies(j, g.my, g.per[1], cj), nk = copies(k, g.mz, g.per[2], ck);
    if (ni * nj * nk == 1) return;
    V3 s{0.0, 0.0, 0.0};
    for (int r = 0; r < nk; r++)
        for (int q = 0; q < nj; q++)
            for (int p = 0; p < ni; p++) {
                const V3 v = ld3(a, g.L(ck[r], cj[q], ci[p]));
                s = V3{s.x + v.x, s.y + v.y, s.z + v.z};
            }
    st3(a, g.L(k, j, i), s);
}

// ucat = M^-1 q at an interior cell, M the rows csi, eta, zet: qbar = M^-T ucat_bar, by Cramer's
// rule on M^T; written for the interior cells (nothing else of qbar is read)
__global__ void k_c2c_adj_solve(const double *ubar, const double *csi, const double *eta, const double *zet,
                                double *qbar, Geo g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1, j = blockIdx.y * blockDim.y + threadIdx.y + 1,
              k = blockIdx.z + 1;
    if (i > g.mx - 2 || j > g.my - 2 || k > g.mz - 2) return;
    const long c = g.L(k, j, i);
    const V3 cs = ld3(csi, c), et = ld3(eta, c), ze = ld3(zet, c);
    // T = M^T: columns csi, eta, zet
    const double t00 = cs.x, t01 = et.x, t02 = ze.x, t10 = cs.y, t11 = et.y, t12 = ze.y, t20 = cs.z, t21 = et.z,
                 t22 = ze.z;
    const V3 r = ld3(ubar, c);
    const double det = t00 * (t11 * t22 - t12 * t21) - t01 * (t10 * t22 - t12 * t20) + t02 * (t10 * t21 - t11 * t20);
    const double d0 = r.x * (t11 * t22 - t12 * t21) - r.y * (t01 * t22 - t02 * t21) + r.z * (t01 * t12 - t02 * t11);
    const double d1 = -r.x * (t10 * t22 - t12 * t20) + r.y * (t00 * t22 - t02 * t20) - r.z * (t00 * t12 - t02 * t10);
    const double d2 = r.x * (t10 * t21 - t11 * t20) - r.y * (t00 * t21 - t01 * t20) + r.z * (t00 * t11 - t01 * t10);
    st3(qbar, c, V3{d0 / det, d1 / det, d2 / det});
}

// q_a of cell c averages the faces c - e_a and c of component a, so face p collects half of qbar_a
// of the cells p and p + e_a (zero outside the interior cells); added with vbar (the owned range of a local
// cotangent) to the global xbar, one thread per owned point.  Bound by memory (96 bytes a point): 29 us at
// 128 x 96 x 64, where clearing qbar, adding to vbar and adding vbar to xbar apart took 48
__global__ void k_c2c_adj_gather(const double *qbar, const double *vbar, double *xbar, Geo g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
    if (i > g.mx - 1 || j > g.my - 1) return;
    const long c = g.L(k, j, i);
    auto in = [](int x, int m) { return x >= 1 && x <= m - 2; };
    const bool I = in(i, g.mx), J = in(j, g.my), K = in(k, g.mz);
    auto q = [&](bool cell, int a, long p) { return cell ? qbar[3 * p + a] : 0.0; };
    const V3 v = ld3(vbar, c);
    double *x = xbar + 3 * gidx(g, k, j, i);
    x[0] = x[0] + (v.x + 0.5 * (q(I && J && K, 0, c) + q(in(i + 1, g.mx) && J && K, 0, c + 1)));
    x[1] = x[1] + (v.y + 0.5 * (q(I && J && K, 1, c) + q(I && in(j + 1, g.my) && K, 1, g.L(k, j + 1, i))));
    x[2] = x[2] + (v.z + 0.5 * (q(I && J && K, 2, c) + q(I && J && in(k + 1, g.mz), 2, g.L(k + 1, j, i))));
}

// Transpose of the ExplicitRhsU face resets on a global vector, with x the flux before them: plane 0 of
// each periodic axis took plane m-2 over the whole owned range of the other two axes (all three
// components), one axis after the other, so a point collects the cotangents of its copies, which keep none;
// then the patches' rule (the same faces as the forward's).  Every point is written by one thread: the copies,
// those with an index 0 on a periodic axis, by their source's
__global__ void __launch_bounds__(256) k_face_resets_adj(double *xbar, const double *x, Geo g, PatchKinds P, Shell S) {
    int q[3];
    if (!shell_point(S, blockIdx.x * blockDim.x + threadIdx.x, q[0], q[1], q[2])) return;
    const int m[3] = {g.mx, g.my, g.mz};
    bool two[3], copy = false;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const bool per = g.per[a] != TOSCA_PERIODIC_NONE;
        copy = copy || (per && q[a] == 0);
        two[a] = per && q[a] == m[a] - 2;
    }
    if (copy) return;
    double s[3] = {0.0, 0.0, 0.0};
    for (int di = 0; di <= two[0]; di++)
        for (int dj = 0; dj <= two[1]; dj++)
            for (int dk = 0; dk <= two[2]; dk++) {
                const long o = 3 * gidx(g, dk ? 0 : q[2], dj ? 0 : q[1], di ? 0 : q[0]);
                for (int a = 0; a < 3; a++) {
                    s[a] = s[a] + xbar[o + a];
                    if (di | dj | dk) xbar[o + a] = 0.0;
                }
            }
    const long o = 3 * gidx(g, q[2], q[1], q[0]);
    const bool in = q[0] <= m[0] - 2 && q[1] <= m[1] - 2 && q[2] <= m[2] - 2;
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
        for (int side = 0; side < 2; side++) {
            if (!in || q[a] != (side ? m[a] - 2 : 0)) continue;
            const int b = P.bc[2 * a + side];
            if (b == TOSCA_BCU_NOSLIP || b == TOSCA_BCU_WALLFUNCTION || b == TOSCA_BCU_SLIP) s[a] = 0.0;
            else if (b == TOSCA_BCU_ZEROGRADIENT) {
                const double v = x[o + a];
                if (side == 0 ? v > 0.0 : v < 0.0) s[a] = 0.0;
            }
        }
        xbar[o + a] = s[a];
    }
}

}  // namespace

void launch_rk3w_update(double *ucont, const double *rhs, double *rhs_o, double a, double b, const Geo &g,
                        hipStream_t s) {
    const long n = 3L * g.mx * g.my * g.mz;
    TOSCA_LAUNCH("k_rk3w_update", k_rk3w_update, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ucont, rhs, rhs_o,
                 a, b, g, n);
}

void launch_rk3w_adj_combine(const double *xbar, double *carry, double *rbar, double a, double b, const Geo &g,
                             hipStream_t s) {
    const long n = 3L * g.mx * g.my * g.mz;
    TOSCA_LAUNCH("k_rk3w_adj_combine", k_rk3w_adj_combine, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, xbar,
                 carry, rbar, a, b, n);
}

// transpose of launch_reset_cell_periodic on a vector field, for the interior cells
void launch_reset_cell_periodic_adj(double *a, const Geo &g, hipStream_t s) {
    // the points that have copies: up to GW from a wrapped end, the first and last interior cells otherwise;
    // over the boundary cells of the other axes too, whose copies are no interior cells', nothing is needed
    const int m[3] = {g.mx, g.my, g.mz};
    int olo[3], ohi[3], clo[3], chi[3];
    for (int q = 0; q < 3; q++) {
        const bool per = g.per[q] != TOSCA_PERIODIC_NONE, wrap = g.per[q] == TOSCA_PERIODIC_WRAP;
        olo[q] = 1; ohi[q] = m[q] - 1;
        clo[q] = min(ohi[q], wrap ? GW : per ? 2 : 1);
        chi[q] = max(clo[q], wrap ? m[q] - GW : per ? m[q] - 2 : m[q] - 1);
    }
    const Shell S = make_shell(olo, ohi, clo, chi);
    if (S.total) TOSCA_LAUNCH("k_ghosts_adj", k_ghosts_adj, dim3((S.total + 255) / 256), dim3(256), 0, s, a, g, S);
}

void launch_c2c_adj(const double *ubar, const tosca_mesh *m, double *qbar, const double *vbar, double *xbar, const Geo &g,
                    hipStream_t s) {
    TOSCA_LAUNCH("k_c2c_adj_solve", k_c2c_adj_solve, dim3((g.mx - 2 + 63) / 64, (g.my - 2 + 3) / 4, g.mz - 2),
                 dim3(64, 4), 0, s, ubar, m->csi, m->eta, m->zet, qbar, g);
    TOSCA_LAUNCH("k_c2c_adj_gather", k_c2c_adj_gather, dim3((g.mx + 63) / 64, (g.my + 3) / 4, g.mz), dim3(64, 4), 0, s, qbar, vbar,
                 xbar, g);
}

// transpose of the ExplicitRhsU face resets y = Pf(Pn(x)) on a global cotangent (x: the state before the resets)
void launch_face_resets_adj(double *xbar, const double *x, const tosca_params *p, const Geo &g, hipStream_t s) {
    const int zero[3] = {0, 0, 0}, own[3] = {g.mx, g.my, g.mz}, lo[3] = {1, 1, 1}, hi[3] = {g.mx - 2, g.my - 2, g.mz - 2};
    const Shell S = make_shell(zero, own, lo, hi);
    TOSCA_LAUNCH("k_face_resets_adj", k_face_resets_adj, dim3((S.total + 255) / 256), dim3(256), 0, s, xbar, x, g, patch_kinds(p), S);
}

}  // namespace tosca
