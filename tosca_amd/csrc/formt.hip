// formt.hip -- FormT (src/solvers/teqn_solvers.c:6-592), the divergence and viscous fluxes of the
// potential-temperature equation and their cell budgets, on gfx950.  Compiled with FP contraction
// off: every face flux is evaluated in the reference's expression order.
//
//   k_formt   the fused i/j/k face loop (teqn_solvers.c:117-481): WENO3 upwinded advective flux and
//             the diffusive flux with the effective diffusivity of the LES closure (nu/Pr, the subgrid
//             diffusivity k_t, or nu_t over the stability-corrected turbulent Prandtl number) and the
//             wall heat flux of thetaWallFunction patches; face 0 of a periodic axis taken as face m-2
//             (resetFacePeriodicFluxesVector, :487-503); the flux budgets of the interior cells times
//             the cell Jacobian (:511-537).  The fluxes never reach memory.
#include "fused.h"

namespace tosca {

namespace {

struct FormTArgs {
    const double *ucont, *t, *nut, *kt;
    const double *icsi, *ieta, *izet, *jcsi, *jeta, *jzet, *kcsi, *keta, *kzet;
    const double *iaj, *jaj, *kaj;
    const double *qI, *qJ;       // wall heat flux [3][mz][my] (i patches), [3][mz][mx] (j patches)
    const double *aj;
    double *rhs;
    double nu, pr, tref, scale;
    int wall[4], mode;
};

// Compute_dscalar_i / _j / _k (src/include/inline.h:3210-3342) with no IBM or overset cells, across the
// face and its two transverse axes: four-point transverse averages, which become two-point one-sided
// averages on the face rows next to a non-periodic boundary edge.  Along a transverse axis (index x of
// 1 .. m-2, point stride st): the offsets of the two rows and the weight.
struct Across { int hi, lo; double w; };
__device__ __forceinline__ Across across(bool edge, int x, int m, int st) {
    const bool top = edge && x == m - 2, bot = edge && x == 1 && !top;
    return Across{top ? 0 : st, bot ? 0 : -st, top || bot ? 0.5 : 0.25};
}

// getFace2Cell4Stencil{Csi,Eta,Zet} (src/include/inline.h:2190-2330): the outer cells of the
// four-cell stencil of face f on an axis with m points
__device__ __forceinline__ void face_stencil(int ptype, int f, int m, int &L, int &R) {
    if (f == 0 || f == m - 2) {
        if (ptype == TOSCA_PERIODIC_COPY) { L = m - 3; R = 2; }
        else if (ptype == TOSCA_PERIODIC_WRAP && f == m - 2) { R = m + 2; L = f - 1; }
        else if (ptype == TOSCA_PERIODIC_WRAP && f == 0) { L = -3; R = f + 2; }
        else if (f == 0) { L = f; R = f + 2; }
        else { L = f - 1; R = f + 1; }
    } else {
        L = f - 1; R = f + 2;
    }
}

// weno3 (src/include/inline.h:5147-5179): third-order WENO face value upwinded on the sign of the
// face flux; the reference squares with pow(x, 2.), here the correctly rounded product
__device__ __forceinline__ double weno3(double f0, double f1, double f2, double f3, double wavespeed) {
    double fL, fC, fR;
    if (wavespeed > 0) { fL = f0; fC = f1; fR = f2; }
    else { fL = f3; fC = f2; fR = f1; }
    const double d0 = 2. / 3., d1 = 1. / 3.;
    const double eps = 1.e-6;
    const double beta0 = (fC - fR) * (fC - fR);
    const double beta1 = (fL - fC) * (fL - fC);
    const double alpha0 = d0 / ((eps + beta0) * (eps + beta0));
    const double alpha1 = d1 / ((eps + beta1) * (eps + beta1));
    const double sumalpha = alpha0 + alpha1;
    const double w0 = alpha0 / sumalpha, w1 = alpha1 / sumalpha;
    const double u0 = (fC * 0.5 + fR * 0.5);
    const double u1 = (-fL * 0.5 + fC * 1.5);
    return w0 * u0 + w1 * u1;
}

// effective diffusivity of a face between cells c and cn (teqn_solvers.c:168-200 and the j / k
// copies): nu/Pr without LES; with LES (nu set to 0) the face-averaged k_t of the models that
// carry one, else nu_t over the turbulent Prandtl number 1 / (1 + 2 l / delta), with the
// stability length l = min(delta, 7.6 nu_t / delta sqrt(T_ref / |g . grad T|)) in stable
// stratification (g . grad T < 0) and l = delta otherwise
enum { KAP_NONE, KAP_KT, KAP_NUT };      // no LES, a model that carries k_t, nu_t over Pr_t
// (ka, kb: k_t or nu_t of the face's two cells)
template <int KAP>
__device__ __forceinline__ double kappa_eff(const FormTArgs &A, double ka, double kb, double ajc, double dtde) {
    if constexpr (KAP == KAP_NONE) return A.nu / A.pr;
    const double nu = 0.0;
    if constexpr (KAP == KAP_KT) {
        const double diff = 0.5 * (ka + kb);
        return (nu / A.pr) + diff;
    }
    const double nut = 0.5 * (ka + kb);
    const double gradTdotG = dtde * (-9.81);
    const double vol = 1. / ajc, delta = vol < 0. ? nan("") : cube_root(vol);      // pow(vol, 1. / 3.)
    double l;
    if (gradTdotG < 0.) {
        const double ls = 7.6 * nut / delta * sqrt(A.tref / fabs(gradTdotG));
        l = delta < ls ? delta : ls;
    }
    else l = delta;
    const double Prt = 1.0 / (1.0 + (2.0 * l / delta));
    return (nu / A.pr) + (nut / Prt);
}

// What a face's flux takes from the cells: theta of the pair and of the stencil's outer cells, the differences
// along the three axes, k_t or nu_t of the pair
struct FaceCells { double T0, T1, L, R, dt[3], ka, kb; };

// The advective (d) and diffusive (v) flux of one face, as the reference's face loop evaluates it
// (teqn_solvers.c:127-246 / 250-370 / 374-478).  Face (i, j, k) of direction DIR lies between cell
// (i, j, k), local index c, and its + neighbour along DIR.
template <int DIR, int KAP>
__device__ __forceinline__ void cell_flux(const FormTArgs &A, const Geo &g, int i, int j, int k, int c, double u, const FaceCells &F,
                                          double &d, double &v) {
    const int f = DIR == 0 ? i : DIR == 1 ? j : k, m = DIR == 0 ? g.mx : DIR == 1 ? g.my : g.mz;
    const double ajc = (DIR == 0 ? A.iaj : DIR == 1 ? A.jaj : A.kaj)[c];
    const V3 cs = ld3(DIR == 0 ? A.icsi : DIR == 1 ? A.jcsi : A.kcsi, c), et = ld3(DIR == 0 ? A.ieta : DIR == 1 ? A.jeta : A.keta, c),
             ze = ld3(DIR == 0 ? A.izet : DIR == 1 ? A.jzet : A.kzet, c);
    d = -u * weno3(F.L, F.T0, F.T1, F.R, u);
    double kap = kappa_eff<KAP>(A, F.ka, F.kb, ajc, F.dt[1]);
    const V3 n = DIR == 0 ? cs : DIR == 1 ? et : ze;
    const double g11 = cs.x * n.x + cs.y * n.y + cs.z * n.z;
    const double g21 = et.x * n.x + et.y * n.y + et.z * n.z;
    const double g31 = ze.x * n.x + ze.y * n.y + ze.z * n.z;
    v = 0.0;
    if constexpr (DIR < 2 && KAP != KAP_NONE) {
        if ((A.wall[2 * DIR] && f == 0) || (A.wall[2 * DIR + 1] && f == m - 2)) {
            const double signQ = (f == 0) ? -1.0 : 1.0;
            const double *q = DIR == 0 ? A.qI : A.qJ;
            const int n1 = DIR == 0 ? g.my : g.mx, pl = g.mz * n1, o = k * n1 + (DIR == 0 ? j : i);
            v = signQ * (q[o] * n.x + q[pl + o] * n.y + q[2 * pl + o] * n.z);
            kap = 0.0;
        }
    }
    v += (g11 * F.dt[0] + g21 * F.dt[1] + g31 * F.dt[2]) * ajc * kap;
}

// the same with the cells' values loaded
template <int DIR, int KAP>
__device__ __forceinline__ void face_flux(const FormTArgs &A, const Geo &g, int i, int j, int k, int c, double &d, double &v) {
    const double *T = A.t, *K = KAP == KAP_KT ? A.kt : A.nut;
    const int x[3] = {i, j, k}, m[3] = {g.mx, g.my, g.mz}, st[3] = {1, g.gxm, g.gxm * g.gym};
    const int f = x[DIR], sd = st[DIR];
    FaceCells F;
    F.T0 = T[c]; F.T1 = T[c + sd];
    const bool edge = f == 0 || f == m[DIR] - 2;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        if (q == DIR) { F.dt[q] = F.T1 - F.T0; continue; }
        const Across a = across(edge && (g.nonper(q) || g.nonper(DIR)), x[q], m[q], st[q]);
        F.dt[q] = (T[c + sd + a.hi] + T[c + a.hi] - T[c + sd + a.lo] - T[c + a.lo]) * a.w;
    }
    int L, R;
    face_stencil(g.per[DIR], f, m[DIR], L, R);
    F.L = T[c + (L - f) * sd]; F.R = T[c + (R - f) * sd];
    F.ka = KAP == KAP_NONE ? 0.0 : K[c]; F.kb = KAP == KAP_NONE ? 0.0 : K[c + sd];
    cell_flux<DIR, KAP>(A, g, i, j, k, c, A.ucont[3 * c + DIR], F, d, v);
}

// the difference along a transverse axis (index x of 1 .. m-2) from the pairs (+ cell, own cell) of the row
// above, the face's own row and the row below: across()'s choice on values
__device__ __forceinline__ double across_of(bool edge, int x, int m, double hp, double h, double op, double o, double lp, double l) {
    const bool top = edge && x == m - 2, bot = edge && x == 1 && !top;
    return ((top ? op : hp) + (top ? o : h) - (bot ? op : lp) - (bot ? o : l)) * (top || bot ? 0.5 : 0.25);
}

// ------------------------------------------------------------------------------------------------
// Face fluxes, their budgets and the cell Jacobian in one launch.  A workgroup of NR rows of 64 points
// marches along k: the i face below a cell comes from the lane before, the j face from the row before
// through LDS (one barrier a plane, two buffers; row 0 only supplies its j faces) and the k face from the
// plane before, in registers.  theta comes from registers too: four loads a point and plane (row j at k+2,
// rows j-1 and j+1 at k+1, row j+2 at k), the others from the planes before and the lanes beside, so that
// lanes 2 .. 61 own cells.  Face 0 of a periodic axis is evaluated as face m-2, which
// resetFacePeriodicFluxesVector copies there.
// Bound by the loads: 296 bytes a point at 4.0 TB/s, 128 registers (four waves a SIMD).  384 x 256 x 128,
// k_t: 1.27 ms as a face kernel that stored both fluxes of every face (0.95), twelve ghost launches on them
// and a budget kernel; 1.06 in one launch with theta loaded for each face (36 loads, whose L1 lines were a
// third of the kernel's); 0.93 so.  nu_t over the turbulent Prandtl number: 1.36, 1.28, 1.05 (with pow() for
// the cube root of the volume its constants, kept in registers across the planes, took 174 registers: 1.35).
// The closure is a template parameter for the same reason.  Rows of 4 measured 0.98.
// rhs = scale ((formMode != 2 ? div budget : 0) + (formMode != 1 ? visc budget : 0)) aj, interior
// cells only (the reference writes nothing else of Rhs)
// ------------------------------------------------------------------------------------------------
constexpr int FT_NR = 8, FT_TI = 60, FT_TJ = FT_NR - 1;

template <int KAP>
__global__ void __launch_bounds__(64 * FT_NR, 4) k_formt(FormTArgs A, Geo g, int kchunk) {
    __shared__ double sJ[2][2][FT_NR][64];             // j-face fluxes (advective, diffusive) of the plane
    const int lane = threadIdx.x, r = __builtin_amdgcn_readfirstlane(threadIdx.y);      // a wave is one row
    const int tile = xcd_tile();                       // j fastest, then i, then the k chunk
    const int bj = tile % gridDim.y, bi = (tile / gridDim.y) % gridDim.x, bk = tile / (gridDim.x * gridDim.y);
    const int i = bi * FT_TI + lane - 1, j = bj * FT_TJ + r;
    const int kb = 1 + bk * kchunk, ke = min(kb + kchunk, g.mz - 1);      // cells [kb, ke)
    const bool per0 = !g.nonper(0), per1 = !g.nonper(1), per2 = !g.nonper(2);
    const bool row = r >= 1 && j <= g.my - 2;          // a row of cells (row 0 and rows past the end: j faces at most)
    const bool cell = lane >= 2 && lane <= 61 && i <= g.mx - 2 && row;
    // the row evaluated (face 0 of a periodic axis: face m-2) and this lane's column, clamped
    const int jf = min(j == 0 && per1 ? g.my - 2 : j, g.my - 2), ia = min(i, g.mx + 1), ic = min(max(i, 0), g.mx - 2), i1 = max(ic, 1);
    const int SJ = g.gxm, SK = g.gxm * g.gym;
    const int t0 = g.L(0, jf, ia), c0 = g.L(0, jf, ic), tE = g.L(0, jf == g.my - 2 && per1 ? (g.per[1] == TOSCA_PERIODIC_COPY ? 2 : g.my + 2) : jf + 2, ia);
    const bool eI = i == 0 || i == g.mx - 2, eJ = jf == 0 || jf == g.my - 2;
    const bool nIJ = g.nonper(0) || g.nonper(1), nIK = g.nonper(0) || g.nonper(2), nJK = g.nonper(1) || g.nonper(2);
    const double *T = A.t, *K = KAP == KAP_KT ? A.kt : A.nut;
    double dKm = 0.0, vKm = 0.0;                       // the k face below the cell
    if (cell) {
        const int kf = (kb == 1 && per2) ? g.mz - 2 : kb - 1;
        face_flux<2, KAP>(A, g, i, j, kf, g.L(kf, j, i), dKm, vKm);
    }
    // theta of the column: own row at planes k-1 .. k+2, row j+1 at k-1 .. k+1, row j-1 at k, k+1
    int t = t0 + kb * SK;
    double a0 = T[t - SK], a1 = T[t], a2 = T[t + SK], b0 = T[t + SJ - SK], b1 = T[t + SJ], m1 = T[t - SJ];
    double kp0 = KAP == KAP_NONE ? 0.0 : K[t];
    for (int k = kb; k < ke; k++) {
        const int buf = k & 1, c = opaque_index(c0 + k * SK);
        t = opaque_index(t0 + k * SK);
        const int kR = k == g.mz - 2 && per2 ? (g.per[2] == TOSCA_PERIODIC_COPY ? 2 : g.mz + 2) : k + 2;
        const double a3 = T[t0 + kR * SK], b2 = T[t + SJ + SK], m2 = T[t - SJ + SK], e = T[tE + k * SK];
        double kpJ = 0.0, kpK = 0.0;
        if constexpr (KAP != KAP_NONE) { kpJ = K[t + SJ]; kpK = K[t + SK]; }
        const V3 u = ld3(A.ucont, c);
        const double a1p = shdn(a1), a1m = shup(a1), b1p = shdn(b1), b1m = shup(b1), a2p = shdn(a2), a2m = shup(a2);
        double dI = 0.0, vI = 0.0, dJ = 0.0, vJ = 0.0, dK = 0.0, vK = 0.0;
        {
            FaceCells F;
            F.T0 = a1; F.T1 = b1;
            F.L = jf == 0 ? a1 : m1;
            F.R = jf == g.my - 2 && !per1 ? b1 : e;
            F.dt[0] = across_of(eJ && nIJ, i, g.mx, b1p, a1p, b1, a1, b1m, a1m);
            F.dt[1] = b1 - a1;
            F.dt[2] = across_of(eJ && nJK, k, g.mz, b2, a2, b1, a1, b0, a0);
            F.ka = kp0; F.kb = kpJ;
            cell_flux<1, KAP>(A, g, i1, jf, k, c, u.y, F, dJ, vJ);
        }
        sJ[buf][0][r][lane] = dJ; sJ[buf][1][r][lane] = vJ;
        if (row) {
            const double a0p = shdn(a0), m1p = shdn(m1), a1pp = shdn(a1p), kpI = shdn(kp0);
            {
                FaceCells F;
                F.T0 = a1; F.T1 = a1p;
                F.L = i == 0 ? a1 : a1m;
                F.R = i == g.mx - 2 ? a1p : a1pp;
                if (per0 && i == g.mx - 2) F.R = T[g.L(k, j, g.per[0] == TOSCA_PERIODIC_COPY ? 2 : g.mx + 2)];
                F.dt[0] = a1p - a1;
                F.dt[1] = across_of(eI && nIJ, j, g.my, b1p, b1, a1p, a1, m1p, m1);
                F.dt[2] = across_of(eI && nIK, k, g.mz, a2p, a2, a1p, a1, a0p, a0);
                F.ka = kp0; F.kb = kpI;
                cell_flux<0, KAP>(A, g, ic, j, k, c, u.x, F, dI, vI);
                // face 0 of a periodic axis: face m-2, out of this row's reach
                if (per0 && i == 0) face_flux<0, KAP>(A, g, g.mx - 2, j, k, g.L(k, j, g.mx - 2), dI, vI);
            }
            {
                FaceCells F;
                const bool eK = k == g.mz - 2;
                F.T0 = a1; F.T1 = a2; F.L = a0;
                F.R = eK && !per2 ? a2 : a3;
                F.dt[0] = across_of(eK && nIK, i, g.mx, a2p, a1p, a2, a1, a2m, a1m);
                F.dt[1] = across_of(eK && nJK, j, g.my, b2, b1, a2, a1, m2, m1);
                F.dt[2] = a2 - a1;
                F.ka = kp0; F.kb = kpK;
                cell_flux<2, KAP>(A, g, i1, j, k, c, u.z, F, dK, vK);
            }
        }
        const double dIm = shup(dI), vIm = shup(vI);
        __syncthreads();
        if (cell) {
            const double dJm = sJ[buf][0][r - 1][lane], vJm = sJ[buf][1][r - 1][lane];
            const double divBudget = dI - dIm + dJ - dJm + dK - dKm, viscBudget = vI - vIm + vJ - vJm + vK - vKm;
            A.rhs[g.G(k, j, i)] = A.scale * ((A.mode != 2 ? divBudget : 0.0) + (A.mode != 1 ? viscBudget : 0.0)) * A.aj[c];
        }
        dKm = dK; vKm = vK;
        a0 = a1; a1 = a2; a2 = a3; b0 = b1; b1 = b2; m1 = m2;
        kp0 = kpK;
    }
}

bool kt_model(int m) {
    return m == TOSCA_LES_AMD || m == TOSCA_LES_DSM || m == TOSCA_LES_DLASI || m == TOSCA_LES_DLASD ||
           m == TOSCA_LES_DPASD || m == TOSCA_LES_BAMD;
}

}  // namespace

namespace {
FormTArgs formt_args(const Geo &g, const tosca_mesh *m, const tosca_params *p, const tosca_teqn_params *tp,
                     const double *ucont, const double *theta, const double *nut, const double *kt) {
    FormTArgs A;
    A.ucont = ucont; A.t = theta; A.nut = nut; A.kt = kt;
    A.icsi = m->icsi; A.ieta = m->ieta; A.izet = m->izet;
    A.jcsi = m->jcsi; A.jeta = m->jeta; A.jzet = m->jzet;
    A.kcsi = m->kcsi; A.keta = m->keta; A.kzet = m->kzet;
    A.iaj = m->iaj; A.jaj = m->jaj; A.kaj = m->kaj;
    A.qI = tp->q_wall_i; A.qJ = tp->q_wall_j;
    A.aj = m->aj; A.rhs = nullptr;
    A.nu = p->nu; A.pr = tp->pr; A.tref = p->t_ref;
    for (int q = 0; q < 4; q++) A.wall[q] = tp->wall_t[q];
    return A;
}
}  // namespace

void formt(const Geo &g, const tosca_mesh *m, const tosca_params *p, const tosca_teqn_params *tp,
           const double *ucont, const double *theta, const double *nut, const double *kt, double *rhs,
           double scale, int mode, hipStream_t s) {
    FormTArgs A = formt_args(g, m, p, tp, ucont, theta, nut, kt);
    A.rhs = rhs; A.scale = scale; A.mode = mode;
    const int ti = (g.mx - 2 + FT_TI - 1) / FT_TI, tj = (g.my - 2 + FT_TJ - 1) / FT_TJ;
    const int kc = plane_chunk(g.mz - 2, ti * tj, CHUNK_FORMT);
    const dim3 grid(ti, tj, (g.mz - 2 + kc - 1) / kc), block(64, FT_NR);
    if (!p->les_active) TOSCA_LAUNCH("k_formt", k_formt<KAP_NONE>, grid, block, 0, s, A, g, kc);
    else if (kt_model(p->les_model)) TOSCA_LAUNCH("k_formt", k_formt<KAP_KT>, grid, block, 0, s, A, g, kc);
    else TOSCA_LAUNCH("k_formt", k_formt<KAP_NUT>, grid, block, 0, s, A, g, kc);
}

}  // namespace tosca
