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
template <int KAP>
__device__ __forceinline__ double kappa_eff(const FormTArgs &A, int c, int cn, double ajc, double dtde) {
    if constexpr (KAP == KAP_NONE) return A.nu / A.pr;
    const double nu = 0.0;
    if constexpr (KAP == KAP_KT) {
        const double diff = 0.5 * (A.kt[c] + A.kt[cn]);
        return (nu / A.pr) + diff;
    }
    const double nut = 0.5 * (A.nut[c] + A.nut[cn]);
    const double gradTdotG = dtde * (-9.81);
    const double delta = pow(1. / ajc, 1. / 3.);
    double l;
    if (gradTdotG < 0.) {
        const double ls = 7.6 * nut / delta * sqrt(A.tref / fabs(gradTdotG));
        l = delta < ls ? delta : ls;
    }
    else l = delta;
    const double Prt = 1.0 / (1.0 + (2.0 * l / delta));
    return (nu / A.pr) + (nut / Prt);
}

// The advective (d) and diffusive (v) flux of one face, as the reference's face loop evaluates it
// (teqn_solvers.c:127-246 / 250-370 / 374-478).  Face (i, j, k) of direction DIR lies between cell
// (i, j, k), local index c, and its + neighbour along DIR.
template <int DIR, int KAP>
__device__ __forceinline__ void face_flux(const FormTArgs &A, const Geo &g, int i, int j, int k, int c, double &d, double &v) {
    const double *T = A.t;
    const int x[3] = {i, j, k}, m[3] = {g.mx, g.my, g.mz}, st[3] = {1, g.gxm, g.gxm * g.gym};
    const int f = x[DIR], sd = st[DIR];
    const double ajc = (DIR == 0 ? A.iaj : DIR == 1 ? A.jaj : A.kaj)[c];
    const V3 cs = ld3(DIR == 0 ? A.icsi : DIR == 1 ? A.jcsi : A.kcsi, c), et = ld3(DIR == 0 ? A.ieta : DIR == 1 ? A.jeta : A.keta, c),
             ze = ld3(DIR == 0 ? A.izet : DIR == 1 ? A.jzet : A.kzet, c);
    const double T0 = T[c], T1 = T[c + sd];
    double dt[3];
    const bool edge = f == 0 || f == m[DIR] - 2;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        if (q == DIR) { dt[q] = T1 - T0; continue; }
        const Across a = across(edge && (g.nonper(q) || g.nonper(DIR)), x[q], m[q], st[q]);
        dt[q] = (T[c + sd + a.hi] + T[c + a.hi] - T[c + sd + a.lo] - T[c + a.lo]) * a.w;
    }
    int L, R;
    face_stencil(g.per[DIR], f, m[DIR], L, R);
    const double u = A.ucont[3 * c + DIR];
    d = -u * weno3(T[c + (L - f) * sd], T0, T1, T[c + (R - f) * sd], u);
    double kap = kappa_eff<KAP>(A, c, c + sd, ajc, dt[1]);
    const V3 n = DIR == 0 ? cs : DIR == 1 ? et : ze;
    const double g11 = cs.x * n.x + cs.y * n.y + cs.z * n.z;
    const double g21 = et.x * n.x + et.y * n.y + et.z * n.z;
    const double g31 = ze.x * n.x + ze.y * n.y + ze.z * n.z;
    v = 0.0;
    if (DIR < 2) {
        if (KAP != KAP_NONE && ((A.wall[DIR < 2 ? 2 * DIR : 0] && f == 0) || (A.wall[DIR < 2 ? 2 * DIR + 1 : 0] && f == m[DIR] - 2))) {
            const double signQ = (f == 0) ? -1.0 : 1.0;
            const double *q = DIR == 0 ? A.qI : A.qJ;
            const int n1 = DIR == 0 ? g.my : g.mx, pl = g.mz * n1, o = k * n1 + (DIR == 0 ? j : i);
            v = signQ * (q[o] * n.x + q[pl + o] * n.y + q[2 * pl + o] * n.z);
            kap = 0.0;
        }
    }
    v += (g11 * dt[0] + g21 * dt[1] + g31 * dt[2]) * ajc * kap;
}

// ------------------------------------------------------------------------------------------------
// Face fluxes, their budgets and the cell Jacobian in one launch.  A workgroup of NR rows of 64 points
// (lane 0 and row 0 only supply their + faces) marches along k: the i face below a cell comes from the
// lane before, the j face from the row before through LDS (one barrier a plane, two buffers) and the k
// face from the plane before, in registers.  Face 0 of a periodic axis is evaluated as face m-2, which
// resetFacePeriodicFluxesVector copies there.
// Bound by the loads: 288 bytes a point at 4.1 TB/s, with about 950 L1 lines a wave and plane (nine vectors
// at a stride of 24 bytes); the closure is a template parameter because the constants of pow(), kept in
// registers across the planes, take a k_t model from 113 registers (four waves a SIMD) to 166 (1.22 ms).
// 384 x 256 x 128, k_t: 1.24 ms as a face kernel that stored both fluxes of every face (0.95), twelve ghost
// launches on them and a budget kernel, 1.06 so; 1.28 against 1.36 with nu_t.  Rows of 4 or 16 measured 1.09
// and 1.10, loads without branches (195 registers) 1.24.
// rhs = scale ((formMode != 2 ? div budget : 0) + (formMode != 1 ? visc budget : 0)) aj, interior
// cells only (the reference writes nothing else of Rhs)
// ------------------------------------------------------------------------------------------------
constexpr int FT_NR = 8, FT_TI = 63, FT_TJ = FT_NR - 1;

template <int KAP>
__global__ void __launch_bounds__(64 * FT_NR) k_formt(FormTArgs A, Geo g, int kchunk) {
    __shared__ double sJ[2][2][FT_NR][64];             // j-face fluxes (advective, diffusive) of the plane
    const int lane = threadIdx.x, r = threadIdx.y;
    const int tile = xcd_tile();                       // j fastest, then i, then the k chunk
    const int bj = tile % gridDim.y, bi = (tile / gridDim.y) % gridDim.x, bk = tile / (gridDim.x * gridDim.y);
    const int i = bi * FT_TI + lane, j = bj * FT_TJ + r;
    const int kb = 1 + bk * kchunk, ke = min(kb + kchunk, g.mz - 1);      // cells [kb, ke)
    const bool colI = i >= 1 && i <= g.mx - 2, colJ = j >= 1 && j <= g.my - 2;
    const bool needI = r >= 1 && colJ && i <= g.mx - 2, needJ = lane >= 1 && colI && j <= g.my - 2;
    const bool cell = lane >= 1 && r >= 1 && colI && colJ;
    const int fi = (i == 0 && !g.nonper(0)) ? g.mx - 2 : i, fj = (j == 0 && !g.nonper(1)) ? g.my - 2 : j;
    double dKm = 0.0, vKm = 0.0;                       // the k face below the cell
    if (cell) {
        const int kf = (kb == 1 && !g.nonper(2)) ? g.mz - 2 : kb - 1;
        face_flux<2, KAP>(A, g, i, j, kf, g.L(kf, j, i), dKm, vKm);
    }
    for (int k = kb; k < ke; k++) {
        const int buf = k & 1, ci = opaque_index(g.L(k, j, fi)), cj = opaque_index(g.L(k, fj, i)), c = opaque_index(g.L(k, j, i));
        double dI = 0.0, vI = 0.0, dJ = 0.0, vJ = 0.0, dK = 0.0, vK = 0.0;
        if (needJ) face_flux<1, KAP>(A, g, i, fj, k, cj, dJ, vJ);
        sJ[buf][0][r][lane] = dJ; sJ[buf][1][r][lane] = vJ;
        if (needI) face_flux<0, KAP>(A, g, fi, j, k, ci, dI, vI);
        if (cell) face_flux<2, KAP>(A, g, i, j, k, c, dK, vK);
        const double dIm = shup(dI), vIm = shup(vI);
        __syncthreads();
        if (cell) {
            const double dJm = sJ[buf][0][r - 1][lane], vJm = sJ[buf][1][r - 1][lane];
            const double divBudget = dI - dIm + dJ - dJm + dK - dKm, viscBudget = vI - vIm + vJ - vJm + vK - vKm;
            A.rhs[g.G(k, j, i)] = A.scale * ((A.mode != 2 ? divBudget : 0.0) + (A.mode != 1 ? viscBudget : 0.0)) *
                                  A.aj[c];
        }
        dKm = dK; vKm = vK;
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
    const int kc = plane_chunk(g.mz - 2, ti * tj, 2 * NUM_CU, 1, 500.0);
    const dim3 grid(ti, tj, (g.mz - 2 + kc - 1) / kc), block(64, FT_NR);
    if (!p->les_active) TOSCA_LAUNCH("k_formt", k_formt<KAP_NONE>, grid, block, 0, s, A, g, kc);
    else if (kt_model(p->les_model)) TOSCA_LAUNCH("k_formt", k_formt<KAP_KT>, grid, block, 0, s, A, g, kc);
    else TOSCA_LAUNCH("k_formt", k_formt<KAP_NUT>, grid, block, 0, s, A, g, kc);
}

}  // namespace tosca
