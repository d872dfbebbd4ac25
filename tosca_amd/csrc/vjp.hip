// vjp.hip -- hand-written adjoint (vector-Jacobian product) of the momentum right-hand side.
//
// Function (no counterpart in the reference; it is the adjoint of the reference's forward path):
//   R(ucont, ucat, theta, Cs) = FormU(ucont, ucat, nu_t; scale, formMode 0) + Buoyancy(theta; b)
//   nu_t = UpdateNut(ucat, Cs): Cs Delta^2 |S(ucat)| at interior cells, UpdateNutBCs ghosts
// with every input a full DMDA local array (ghost cells are inputs too) and R on the owned faces.
// Given the cotangent Rbar, the kernels accumulate ucont_bar, ucat_bar, theta_bar, Cs_bar, the
// transpose of each forward stage in reverse order:
//   k_vjp_fp      face dot (ueqn_solvers.c:1006-1035) -> fpbar per interior cell (a gather: the
//                 cell's own faces, the faces of its lower neighbours, and the ghost m-1 aliases:
//                 cell 1 on a periodic axis, the copied cell m-2 otherwise)
//   k_vjp_march   the interior faces: cell divergence (ueqn_solvers.c:871-993) -> face-flux cotangent, then
//                 the convective flux (central / QUICK, inline.h:4314-4324, 5089-5109) -> ucont_bar and its
//                 ucat cotangent, the viscous flux (ueqn_solvers.c:184-216...) -> the cotangents of its nine
//                 derivatives (Compute_du_i/j/k, inline.h:2748-2931) and of nu_eff; the ucat cotangents
//                 summed per row of points, marching along k.  The launch's last workgroups take the
//                 boundary faces, whose stencils are one-sided or clipped: a scatter (atomics)
//   k_vjp_finish  nu_t = Cs Delta^2 |S| (les.c:2510-2514), with the UpdateNutBCs ghosts
//                 (boundary.c:2812-2917) transposed -> Cs_bar and the |S| path (Compute_du_dxyz /
//                 Compute_du_center, inline.h:3344-3418, 3635-3663), added to the row sums -> ucat_bar;
//                 theta_bar from Buoyancy (ueqn_sources.c:2812-2870).  k_vjp_sum: the row sums alone
// The forward intermediates the adjoint needs (nu_t, the face gradients, the interpolated face
// velocities) are recomputed from the inputs instead of being stored by the forward pass.
#include <type_traits>

#include "fused.h"

namespace tosca {

namespace {

__device__ __forceinline__ void aadd(double *p, double v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void aadd(float *p, double v) { unsafeAtomicAdd(p, float(v)); }
template <class T>
__device__ __forceinline__ void aadd3(T *p, int c, V3 v) {
    aadd(p + 3 * c, v.x);
    aadd(p + 3 * c + 1, v.y);
    aadd(p + 3 * c + 2, v.z);
}
__device__ __forceinline__ V3 sc3(double s, V3 v) { return V3{s * v.x, s * v.y, s * v.z}; }
__device__ __forceinline__ V3 add3v(V3 a, V3 b) { return V3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ double dot3(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// w * (p0 + p1 - m0 - m1): adjoint of the four-point differences of Compute_du_*
template <class T>
__device__ __forceinline__ void scat4(T *ub, int p0, int p1, int m0, int m1, double w, V3 gb) {
    const V3 a = sc3(w, gb), b = sc3(-w, gb);
    aadd3(ub, p0, a); aadd3(ub, p1, a); aadd3(ub, m0, b); aadd3(ub, m1, b);
}
template <class T>
__device__ __forceinline__ void scat2(T *ub, int p, int m, double w, V3 gb) {
    aadd3(ub, p, sc3(w, gb)); aadd3(ub, m, sc3(-w, gb));
}

// Cotangents of the nine curvilinear derivatives, grouped by derivative direction: gc = (dudc,
// dvdc, dwdc), ge = (dude, ...), gz = (dudz, ...).  Adjoint of Compute_du_i (same branches).
template <class T>
__device__ void du_i_adj(const Geo &g, T *ub, int i, int j, int k, V3 gc, V3 ge, V3 gz) {
    const bool iN = g.nonper(0), jN = g.nonper(1), kN = g.nonper(2);
    scat2(ub, g.L(k, j, i + 1), g.L(k, j, i), 1.0, gc);
    const bool ib = (i == 0 || i == g.mx - 2);
    if (j == g.my - 2 && ib && (jN || iN)) scat4(ub, g.L(k, j, i + 1), g.L(k, j, i), g.L(k, j - 1, i + 1), g.L(k, j - 1, i), 0.5, ge);
    else if (j == 1 && ib && (jN || iN)) scat4(ub, g.L(k, j + 1, i + 1), g.L(k, j + 1, i), g.L(k, j, i + 1), g.L(k, j, i), 0.5, ge);
    else scat4(ub, g.L(k, j + 1, i + 1), g.L(k, j + 1, i), g.L(k, j - 1, i + 1), g.L(k, j - 1, i), 0.25, ge);
    if (k == g.mz - 2 && ib && (kN || iN)) scat4(ub, g.L(k, j, i + 1), g.L(k, j, i), g.L(k - 1, j, i + 1), g.L(k - 1, j, i), 0.5, gz);
    else if (k == 1 && ib && (kN || iN)) scat4(ub, g.L(k + 1, j, i + 1), g.L(k + 1, j, i), g.L(k, j, i + 1), g.L(k, j, i), 0.5, gz);
    else scat4(ub, g.L(k + 1, j, i + 1), g.L(k + 1, j, i), g.L(k - 1, j, i + 1), g.L(k - 1, j, i), 0.25, gz);
}

// adjoint of Compute_du_j
template <class T>
__device__ void du_j_adj(const Geo &g, T *ub, int i, int j, int k, V3 gc, V3 ge, V3 gz) {
    const bool iN = g.nonper(0), jN = g.nonper(1), kN = g.nonper(2);
    const bool jb = (j == 0 || j == g.my - 2);
    if (i == g.mx - 2 && jb && (iN || jN)) scat4(ub, g.L(k, j + 1, i), g.L(k, j, i), g.L(k, j + 1, i - 1), g.L(k, j, i - 1), 0.5, gc);
    else if (i == 1 && jb && (iN || jN)) scat4(ub, g.L(k, j + 1, i + 1), g.L(k, j, i + 1), g.L(k, j + 1, i), g.L(k, j, i), 0.5, gc);
    else scat4(ub, g.L(k, j + 1, i + 1), g.L(k, j, i + 1), g.L(k, j + 1, i - 1), g.L(k, j, i - 1), 0.25, gc);
    scat2(ub, g.L(k, j + 1, i), g.L(k, j, i), 1.0, ge);
    if (k == g.mz - 2 && jb && (kN || jN)) scat4(ub, g.L(k, j + 1, i), g.L(k, j, i), g.L(k - 1, j + 1, i), g.L(k - 1, j, i), 0.5, gz);
    else if (k == 1 && jb && (kN || jN)) scat4(ub, g.L(k + 1, j + 1, i), g.L(k + 1, j, i), g.L(k, j + 1, i), g.L(k, j, i), 0.5, gz);
    else scat4(ub, g.L(k + 1, j + 1, i), g.L(k + 1, j, i), g.L(k - 1, j + 1, i), g.L(k - 1, j, i), 0.25, gz);
}

// adjoint of Compute_du_k
template <class T>
__device__ void du_k_adj(const Geo &g, T *ub, int i, int j, int k, V3 gc, V3 ge, V3 gz) {
    const bool iN = g.nonper(0), jN = g.nonper(1), kN = g.nonper(2);
    const bool kb = (k == 0 || k == g.mz - 2);
    if (i == g.mx - 2 && kb && (iN || kN)) scat4(ub, g.L(k + 1, j, i), g.L(k, j, i), g.L(k + 1, j, i - 1), g.L(k, j, i - 1), 0.5, gc);
    else if (i == 1 && kb && (iN || kN)) scat4(ub, g.L(k + 1, j, i + 1), g.L(k, j, i + 1), g.L(k + 1, j, i), g.L(k, j, i), 0.5, gc);
    else scat4(ub, g.L(k + 1, j, i + 1), g.L(k, j, i + 1), g.L(k + 1, j, i - 1), g.L(k, j, i - 1), 0.25, gc);
    if (j == g.my - 2 && kb && (jN || kN)) scat4(ub, g.L(k + 1, j, i), g.L(k, j, i), g.L(k + 1, j - 1, i), g.L(k, j - 1, i), 0.5, ge);
    else if (j == 1 && kb && (jN || kN)) scat4(ub, g.L(k + 1, j + 1, i), g.L(k, j + 1, i), g.L(k + 1, j, i), g.L(k, j, i), 0.5, ge);
    else scat4(ub, g.L(k + 1, j + 1, i), g.L(k, j + 1, i), g.L(k + 1, j - 1, i), g.L(k, j - 1, i), 0.25, ge);
    scat2(ub, g.L(k + 1, j, i), g.L(k, j, i), 1.0, gz);
}

// T: type of the flow fields (ucont, ucat, nu_t) and of their cotangents; P: storage type of what
// passes between the kernels (fpbar, the nu_eff cotangents, the row sums).  The cotangent arithmetic
// is FP64 in both forms.
template <class T, class P>
struct VjpArgs {
    const T *ucont, *ucat, *nut;
    T *nut_w;           // where k_vjp_pre writes the recomputed nu_t (the array nut reads)
    const double *cs, *rbar;
    const double *csi, *eta, *zet, *icsi, *ieta, *izet, *jcsi, *jeta, *jzet, *kcsi, *keta, *kzet;
    const double *aj, *iaj, *jaj, *kaj;
    P *fpbar;
    T *vbar, *ubar, *tbar;
    double *csbar;
    double *nutbar_acc; // nu_t given as an input: its cotangent is accumulated here (local)
    P *nueb[3];         // per face direction: cotangent of nu_eff at each face (n values)
    P *rows;            // ucat cotangents summed per row: own, and for rows of other workgroups jp, jm, jpp (n vectors each)
    double *tb;         // theta cotangents summed per row: the row's own, row j+1's (n values each)
    long n;
    double scale, bscale, tRef, nu;
    int quick, les;
    int bc_u[6], bc_nut[6];
};

template <class A_>
__device__ __forceinline__ V3 cellS(const A_ &A, int q, int c) {
    return ld3(q == 0 ? A.csi : (q == 1 ? A.eta : A.zet), c);
}
template <class A_>
__device__ __forceinline__ double faceA(const A_ &A, int q, int c) {
    return (q == 0 ? A.iaj : (q == 1 ? A.jaj : A.kaj))[c];
}
template <class T>
__device__ __forceinline__ Grad grad64(const GradT<T> &a) {
    return Grad{double(a.dudc), double(a.dvdc), double(a.dwdc), double(a.dude), double(a.dvde), double(a.dwde),
                double(a.dudz), double(a.dvdz), double(a.dwdz)};
}
template <class P>
__device__ __forceinline__ void stp3(P *p, int c, V3 v) { p[3 * c] = P(v.x); p[3 * c + 1] = P(v.y); p[3 * c + 2] = P(v.z); }
template <class P>
__device__ __forceinline__ V3 ldp3(const P *p, int c) { return V3{double(p[3 * c]), double(p[3 * c + 1]), double(p[3 * c + 2])}; }

}  // namespace

// zeroes the outer layers of several local arrays in one launch: blockIdx.z selects the array (words 4-byte
// words per point, w layers from either side, ghosts included), blockIdx.y the side
struct ZeroShells { unsigned *p[8]; int words[8], w[8], n; };
__global__ void __launch_bounds__(256) k_vjp_zero_shells(ZeroShells Z, Geo g) {
    const int q = blockIdx.z, side = blockIdx.y, w = Z.w[q], words = Z.words[q];
    // low / high k slabs over the whole planes, low / high j slabs between them, low / high i slabs between those
    int i0 = 0, j0 = 0, k0 = 0, ni = g.gxm, nj = g.gym, nk = g.gzm;
    if (side < 2) { k0 = side ? g.gzm - w : 0; nk = w; }
    else {
        k0 = w; nk = g.gzm - 2 * w;
        if (side < 4) { j0 = side == 3 ? g.gym - w : 0; nj = w; }
        else { j0 = w; nj = g.gym - 2 * w; i0 = side == 5 ? g.gxm - w : 0; ni = w; }
    }
    if (nj <= 0 || nk <= 0) return;
    // (on an axis shorter than 2 w the two slabs overlap)
    const int row = ni * words, tot = row * nj * nk;
    unsigned *p = Z.p[q];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < tot; t += gridDim.x * blockDim.x) {
        const int e = t % row, l = t / row;
        p[(((long)(k0 + l / nj) * g.gym + (j0 + l % nj)) * g.gxm + i0) * words + e] = 0u;
    }
}

// fpbar of interior cell (i, j, k) (a gather; no atomics); S: its csi, eta, zet
template <class T, class P>
__device__ __forceinline__ void fp_cell(const VjpArgs<T, P> &A, const Geo &g, int i, int j, int k, const V3 *S) {
    const int idx[3] = {i, j, k}, m[3] = {g.mx, g.my, g.mz};
    const int c = g.L(k, j, i);
    V3 fb{0, 0, 0};
    for (int q = 0; q < 3; q++) {
        const int dq[3] = {q == 0, q == 1, q == 2};
        const V3 Sc = S[q];
        // face q of this cell (this cell on the left)
        double w = A.scale * faceA(A, q, c) * 0.5 * A.rbar[3 * g.G(k, j, i) + q];
        fb = add3v(fb, sc3(w, Sc));
        // face q of the lower neighbour (this cell on the right)
        if (idx[q] >= 2) {
            const int kk = k - dq[2], jj = j - dq[1], ii = i - dq[0];
            const double w2 = A.scale * faceA(A, q, g.L(kk, jj, ii)) * 0.5 * A.rbar[3 * g.G(kk, jj, ii) + q];
            fb = add3v(fb, sc3(w2, Sc));
        }
        // the ghost cell m-1 to the right of face m-2 carries fp of cell 1 (periodic) or of m-2
        if (g.per[q] != TOSCA_PERIODIC_NONE && idx[q] == 1) {
            int t[3] = {i, j, k};
            t[q] = m[q] - 2;
            const int cf = g.L(t[2], t[1], t[0]);
            t[q] = m[q] - 1;
            const V3 Sg = cellS(A, q, g.L(t[2], t[1], t[0]));
            t[q] = m[q] - 2;
            const double w3 = A.scale * faceA(A, q, cf) * 0.5 * A.rbar[3 * g.G(t[2], t[1], t[0]) + q];
            fb = add3v(fb, sc3(w3, Sg));
        }
        if (g.per[q] == TOSCA_PERIODIC_NONE && idx[q] == m[q] - 2) {
            int t[3] = {i, j, k};
            t[q] = m[q] - 1;
            const V3 Sg = cellS(A, q, g.L(t[2], t[1], t[0]));
            fb = add3v(fb, sc3(w, Sg));
        }
    }
    stp3(A.fpbar, c, fb);
}

// fpbar at every interior cell
template <class T, class P>
__global__ void __launch_bounds__(256) k_vjp_fp(VjpArgs<T, P> A, Geo g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1, j = blockIdx.y * blockDim.y + threadIdx.y + 1,
              k = blockIdx.z + 1;
    if (i > g.mx - 2 || j > g.my - 2 || k > g.mz - 2) return;
    const int c = g.L(k, j, i);
    const V3 S[3] = {ld3(A.csi, c), ld3(A.eta, c), ld3(A.zet, c)};
    fp_cell(A, g, i, j, k, S);
}

// fpbar and the recomputed nu_t = Cs Delta^2 |S| (UpdateNut's interior, as k_nut_fused forms it,
// les.c:2510-2514) of every interior cell, from one load of its csi, eta, zet
template <class T, class P>
__global__ void __launch_bounds__(256) k_vjp_pre(VjpArgs<T, P> A, Geo g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1, j = blockIdx.y * blockDim.y + threadIdx.y + 1,
              k = blockIdx.z + 1;
    if (i > g.mx - 2 || j > g.my - 2 || k > g.mz - 2) return;
    const int c = g.L(k, j, i);
    const V3 S[3] = {ld3(A.csi, c), ld3(A.eta, c), ld3(A.zet, c)};
    const double a = A.aj[c];
    const double Sm = strain_mag(du_dxyz(cvt3<T>(S[0]), cvt3<T>(S[1]), cvt3<T>(S[2]), T(a), du_center(g, A.ucat, i, j, k)));
    const double filter = cube_root(1. / a);
    A.nut_w[c] = T(A.cs[c] * (filter * filter) * Sm);
    fp_cell(A, g, i, j, k, S);
}

// ------------------------------------------------------------------------------------------------
// The two boundary faces per line (the only ones with the one-sided and clipped stencils): the flux
// cotangent, ucont_bar, the nu_eff cotangent, and a scatter into ucat_bar.  About 39 atomics a face and
// three components, at what the L2 takes; the faces run as the last workgroups of the marching launch,
// where they fill its last wave (the 192 x 192 x 128 hill: 0.06 ms there, 0.13 in a launch of their own,
// 0.11 as the first workgroups).
// ------------------------------------------------------------------------------------------------
// one face of direction DIR: x = (i, j, k) its index point, f = x[DIR] = 0 or m-2, the other two
// in 1 .. m-2
template <int DIR, class T, class P>
__device__ __forceinline__ void face_adj(const VjpArgs<T, P> &A, const Geo &g, const int *x) {
    const int m[3] = {g.mx, g.my, g.mz};
    const int f = x[DIR];
    const bool per = g.per[DIR] != TOSCA_PERIODIC_NONE;
    if (per && f == 0) return;                     // face 0 of a periodic axis is face m-2
    const int i = x[0], j = x[1], k = x[2];
    const int c = g.L(k, j, i);
    const int up = (DIR == 0) ? g.L(k, j, i + 1) : (DIR == 1) ? g.L(k, j + 1, i) : g.L(k + 1, j, i);
    // cotangent of the face flux: + fp of the left cell, - fp of the right cell (interior cells)
    V3 Fb{0, 0, 0};
    if (f >= 1) Fb = add3v(Fb, ldp3(A.fpbar, c));
    if (f + 1 <= m[DIR] - 2) Fb = add3v(Fb, sc3(-1.0, ldp3(A.fpbar, up)));
    if (per && f == m[DIR] - 2) {                  // face 0 aliases this face: it is cell 1's left face
        int t[3] = {i, j, k};
        t[DIR] = 1;
        Fb = add3v(Fb, sc3(-1.0, ldp3(A.fpbar, g.L(t[2], t[1], t[0]))));
    }
    const T *u = A.ucat;
    // ---- convective: div = -V * u_face ---------------------------------------------------------
    const T VT = A.ucont[3 * c + DIR];
    const double V = double(VT);
    const V3 cv = sc3(-V, Fb);
    if (A.quick) {
        int L, R;
        face2cell4(g.per[DIR], f, m[DIR], L, R);
        int xl[3] = {i, j, k}, xr[3] = {i, j, k};
        xl[DIR] = L; xr[DIR] = R;
        const int cLL = g.L(xl[2], xl[1], xl[0]), cRR = g.L(xr[2], xr[1], xr[0]);
        const V3 uf = cvt3<double>(quick(ld3(u, cLL), ld3(u, c), ld3(u, up), ld3(u, cRR), VT));
        A.vbar[3 * c + DIR] = T(-dot3(Fb, uf));
        // d/dfU = 1/2 + 2/8, d/dfD = 1/2 - 1/8, d/dfUU = -1/8
        if (V > 0) { aadd3(A.ubar, c, sc3(0.75, cv)); aadd3(A.ubar, up, sc3(0.375, cv)); aadd3(A.ubar, cLL, sc3(-0.125, cv)); }
        else { aadd3(A.ubar, up, sc3(0.75, cv)); aadd3(A.ubar, c, sc3(0.375, cv)); aadd3(A.ubar, cRR, sc3(-0.125, cv)); }
    } else {
        const Vec3<T> a0 = ld3(u, c), a1 = ld3(u, up);
        const V3 uf{double(T(0.5) * (a0.x + a1.x)), double(T(0.5) * (a0.y + a1.y)), double(T(0.5) * (a0.z + a1.z))};
        A.vbar[3 * c + DIR] = T(-dot3(Fb, uf));
        aadd3(A.ubar, c, sc3(0.5, cv));
        aadd3(A.ubar, up, sc3(0.5, cv));
    }
    // ---- viscous ------------------------------------------------------------------------------------
    double nuEff = A.nu;
    bool dep = false;                               // nu_eff depends on nu_t
    if (A.les) {
        const int bl = A.bc_u[2 * DIR], br = A.bc_u[2 * DIR + 1];
        if (DIR < 2 && ((bl == TOSCA_BCU_WALLFUNCTION && f == 0) || (br == TOSCA_BCU_WALLFUNCTION && f == m[DIR] - 2))) {
            nuEff = A.nu;
        } else if ((bl == TOSCA_BCU_SLIP && f == 0) || (br == TOSCA_BCU_SLIP && f == m[DIR] - 2)) {
            nuEff = 0.0;
        } else {
            nuEff = A.nu + 0.5 * (double(A.nut[c]) + double(A.nut[up]));
            dep = true;
        }
    }
    const double *fcp = (DIR == 0) ? A.icsi : (DIR == 1) ? A.jcsi : A.kcsi;
    const double *fep = (DIR == 0) ? A.ieta : (DIR == 1) ? A.jeta : A.keta;
    const double *fzp = (DIR == 0) ? A.izet : (DIR == 1) ? A.jzet : A.kzet;
    const double *fap = (DIR == 0) ? A.iaj : (DIR == 1) ? A.jaj : A.kaj;
    const V3 fc = ld3(fcp, c), fe = ld3(fep, c), fz = ld3(fzp, c);
    const double ajc = fap[c];
    double nb = 0.0;
    if (dep) {
        const Grad gr = grad64((DIR == 0) ? du_i(g, u, i, j, k) : (DIR == 1) ? du_j(g, u, i, j, k) : du_k(g, u, i, j, k));
        nb = dot3(Fb, visc_flux(gr, fc, fe, fz, DIR, ajc, 1.0));
    }
    A.nueb[DIR][c] = P(nb);
    // visc_m = a nu (g_X1 d_X u_m + (M_X . d_X u) n_m) summed over X = csi, eta, zet
    const V3 nrm = (DIR == 0) ? fc : (DIR == 1) ? fe : fz;
    const double g11 = dot3(fc, nrm), g21 = dot3(fe, nrm), g31 = dot3(fz, nrm);
    const V3 Fa = sc3(ajc * nuEff, Fb);
    auto gx = [&](double gX1, V3 MX) {
        const double d = dot3(MX, Fa);
        return V3{gX1 * Fa.x + d * nrm.x, gX1 * Fa.y + d * nrm.y, gX1 * Fa.z + d * nrm.z};
    };
    const V3 gc = gx(g11, fc), ge = gx(g21, fe), gz = gx(g31, fz);
    if (nuEff != 0.0) {
        if (DIR == 0) du_i_adj(g, A.ubar, i, j, k, gc, ge, gz);
        else if (DIR == 1) du_j_adj(g, A.ubar, i, j, k, gc, ge, gz);
        else du_k_adj(g, A.ubar, i, j, k, gc, ge, gz);
    }
}

// thread t of the boundary workgroups: face set t / nmax (direction, low or high side), point t % nmax of it
template <class T, class P>
__device__ __forceinline__ void boundary_face(const VjpArgs<T, P> &A, const Geo &g, int t, int nmax) {
    const int set = t / nmax, d = set / 2, m[3] = {g.mx, g.my, g.mz};
    if (set >= 6) return;
    const int n1 = d == 0 ? g.my : g.mx, n2 = d == 2 ? g.my : g.mz;      // transverse sizes, fastest first
    const int a = t % nmax % n1, b = t % nmax / n1;
    if (a < 1 || a > n1 - 2 || b < 1 || b > n2 - 2) return;
    const int f = set % 2 ? m[d] - 2 : 0;
    const int x[3] = {d == 0 ? f : a, d == 0 ? a : d == 1 ? f : b, d == 2 ? f : b};
    if (d == 0) face_adj<0>(A, g, x);
    else if (d == 1) face_adj<1>(A, g, x);
    else face_adj<2>(A, g, x);
}

// ------------------------------------------------------------------------------------------------
// Interior faces (1 <= f <= m-3 along the face direction), marching along k: ucont_bar, the nu_eff
// cotangents and the ucat cotangents of their regular stencils.
//
// A wave is one row j of 64 points along i and steps through the planes; lane 0 is point i0 - 2, and the
// 60 lanes 2 .. 61 own their cell (a cell collects from the faces i-2 .. i+1).  Each plane the thread evaluates the i, j and k face of its point: the
// convective cotangent cv = -V Fbar and the cotangents gc, ge, gz of the three derivative vectors.  A
// face contributes to the cells
//   normal derivative        left -gn, right +gn
//   convective interpolation left and right (QUICK: left 3/4 or 3/8, right 3/8 or 3/4, and -1/8 of the
//                            cell upwind of the pair; the other end takes nothing, by selection, so that a value
//                            that is not finite reaches the cells of the stencil alone)
//   transverse derivatives   for both cells of the pair: +g/4 one up, -g/4 one down the transverse axis
// and these are added where they land: along i by lane shifts, along k in the accumulators of four
// planes, and what goes to the neighbouring rows, `jp` for row j+1, `jm` for row j-1 and (QUICK) `jpp` for row
// j+2, through LDS where that row is one of the workgroup's four (one barrier a plane) and to memory where it
// is not: per point the row's own sum `own` and, at the workgroup's ends, jp of its last row, jm of its first,
// jpp of its last two, on average 4.5 values (QUICK: 6) instead of the 36 of three face packets.  k_vjp_finish adds the
// rows.  Buoyancy's theta cotangent comes along, since its icsi.z, jeta.z, kzet.z are loaded here.
//
// Bound by memory: 456 bytes a point in FP64 (nine metric vectors 216, row sums 48), 755 moved on the hill below
// (4.2 TB/s), since a wave's 64 points end within cache lines, 4 of them overlap and a chunk of planes loads 3
// more.  The registers (two waves a SIMD) hold the sums of four planes; the row sums and ucont_bar are
// written as whole vectors, since stores of 8 of 24 bytes cost a pass over the line each.  Against a launch
// that wrote the three packets of every face and a cell kernel that gathered them: the adjoint of the
// 192 x 192 x 128 hill (FP64, QUICK) 2.60 -> 1.48 ms, of which this kernel is 0.84, and of the 384 x 256 x 96
// box (mixed, central) 3.69 -> 1.94, of which 1.00.  Without the exchange in LDS every row's sums went to
// memory: 1.52 and 2.06 (this kernel 0.82 and 1.03, k_vjp_finish 0.43 and 0.63 for 0.38 and 0.54); with
// workgroups of eight rows 1.47 and 1.95, but 0.16 for 0.14 on the 128 x 96 x 64 grid, which they do not fill.
constexpr int VM_NR = 4;         // rows of a workgroup
template <class T, class P, bool QUICK>
__global__ void __launch_bounds__(64 * VM_NR, 2) k_vjp_march(VjpArgs<T, P> A, Geo g, int kchunk, int ti, int tj, int nbnd, int nmax) {
    // per row of the workgroup: what it hands to the row above (jp, of plane t-1), to the row below (jm) and to
    // the second row above (jpp), both of plane t and read a plane step later
    __shared__ double sP[2][VM_NR][3][64], sM[3][VM_NR][3][64], sQ[QUICK ? 3 : 1][VM_NR][3][64];
    const int lane = threadIdx.x, r = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int nm = gridDim.x - nbnd;
    if (blockIdx.x >= nm) {
        boundary_face(A, g, ((blockIdx.x - nm) * VM_NR + r) * 64 + lane, nmax);
        return;
    }
    const int tile = xcd_tile(blockIdx.x, nm);      // j fastest, then i, then the k chunk
    const int bj = tile % tj, bi = (tile / tj) % ti, bk = tile / (ti * tj);
    const int jt = 1 + bj * VM_NR + r, i = bi * 60 + lane - 2, j = min(jt, g.my - 2);
    const bool rowOk = jt <= g.my - 2;                 // rows past the end hand out zeros
    const int kb = bk * kchunk, ke = min(kb + kchunk, g.mz);     // cells [kb, ke)
    const int ia = min(max(i, 0), g.mx - 1);
    const int SJ = g.gxm, SK = g.gxm * g.gym, c0 = g.L(0, j, ia);
    const bool mine = lane >= 2 && lane < 62 && i < g.mx && rowOk;
    const bool cellI = i >= 1 && i <= g.mx - 2 && rowOk;
    const bool okJ0 = cellI && j <= g.my - 3;
    const long n = A.n;
    P *own = A.rows, *jp = A.rows + 3 * n, *jm = A.rows + 6 * n, *jpp = A.rows + 9 * n;
    auto up = [](V3 v) { return shup3(v); };           // the value of lane - 1
    auto dn = [](V3 v) { return shdn3(v); };           // the value of lane + 1
    auto sel = [](bool ok, V3 v) { return V3{ok ? v.x : 0.0, ok ? v.y : 0.0, ok ? v.z : 0.0}; };
    const V3 Z{0, 0, 0};
    // sums of the cells of planes t-1 .. t+2 of this row, of planes t-1 .. t+1 for row j+1, the k face's
    // transverse-j cotangent of plane t-1, and the k face's theta cotangent of plane t-1
    V3 a0 = Z, a1 = Z, a2 = Z, a3 = Z, p0 = Z, p1 = Z, p2 = Z, tk = Z;
    double hk = 0.0;
    auto put = [&](double (&d)[VM_NR][3][64], V3 v) { d[r][0][lane] = v.x; d[r][1][lane] = v.y; d[r][2][lane] = v.z; };
    auto from = [&](const double (&d)[VM_NR][3][64], int q) { return V3{d[q][0][lane], d[q][1][lane], d[q][2][lane]}; };
    int slot = 0, last = 2;                            // of planes t and t-1 in sM and sQ
    for (int t = kb - 2; t <= ke; t++) {
        const int tc = min(max(t, 0), g.mz - 1);
        const int c = opaque_index(c0 + tc * SK);
        const bool cell = cellI && t >= 1 && t <= g.mz - 2;      // an interior cell (its + faces exist)
        const bool face = t >= kb && t < ke && mine;             // this thread's faces are written
        const bool okI = cell && i <= g.mx - 3, okJ = cell && okJ0, okK = cell && t <= g.mz - 3;
        const V3 fb = ldp3(A.fpbar, c), fbj = ldp3(A.fpbar, c + SJ), fbk = ldp3(A.fpbar, c + SK), fbi = dn(fb);
        T n0 = T(0), nj = T(0), nk = T(0), ni = T(0);
        if (A.les) { n0 = A.nut[c]; nj = A.nut[c + SJ]; nk = A.nut[c + SK]; ni = shdn(n0); }
        const Vec3<T> V = ld3(A.ucont, c);
        const Vec3<T> u = ld3(A.ucat, c), uj = ld3(A.ucat, c + SJ), ujm = ld3(A.ucat, c - SJ), uk = ld3(A.ucat, c + SK),
                      ukm = ld3(A.ucat, c - SK);
        // (lane shifts stay outside the branches: they read lanes that may not take them)
        const Vec3<T> ui = shdn3(u), uii = shdn3(ui), uim = shup3(u), uji = shdn3(uj), uki = shdn3(uk);
        const T q4 = T(0.25);
        auto four = [&](Vec3<T> a, Vec3<T> b, Vec3<T> m, Vec3<T> o) {
            return V3{double((a.x + b.x - m.x - o.x) * q4), double((a.y + b.y - m.y - o.y) * q4),
                      double((a.z + b.z - m.z - o.z) * q4)};
        };
        auto diff = [&](Vec3<T> a, Vec3<T> b) { return V3{double(a.x - b.x), double(a.y - b.y), double(a.z - b.z)}; };
        // one face: flux cotangent F, normal flux W, derivative vectors d[0..2], face metrics; returns the
        // nu_eff cotangent and writes cv and the cotangents G of the three derivative vectors
        auto adj = [&](auto dir, bool ok, V3 F, double W, const V3 (&d)[3], double nuEff, V3 fc, V3 fe, V3 fz, double ajc, V3 &cv,
                       V3 (&G)[3]) {
            constexpr int DIR = decltype(dir)::value;
            cv = sc3(-W, F);
            double nb = 0.0;
            if (A.les) {
                const Grad gr{d[0].x, d[0].y, d[0].z, d[1].x, d[1].y, d[1].z, d[2].x, d[2].y, d[2].z};
                nb = dot3(F, visc_flux(gr, fc, fe, fz, DIR, ajc, 1.0));
            }
            // visc_m = a nu (g_X1 d_X u_m + (M_X . d_X u) n_m) summed over X = csi, eta, zet
            const V3 M[3] = {fc, fe, fz};
            const V3 nrm = M[DIR], Fa = sc3(ok ? ajc * nuEff : 0.0, F);
#pragma unroll
            for (int X = 0; X < 3; X++) {
                const double gX = dot3(M[X], nrm), s = dot3(M[X], Fa);
                G[X] = sel(ok, V3{gX * Fa.x + s * nrm.x, gX * Fa.y + s * nrm.y, gX * Fa.z + s * nrm.z});
            }
            return ok ? nb : 0.0;
        };
        // face value of u for ucont_bar, and the weights of the left and right cell and (QUICK) the cells beyond
        auto face_u = [&](Vec3<T> m1, Vec3<T> l, Vec3<T> r, Vec3<T> r2, T W) {
            if constexpr (QUICK) return cvt3<double>(quick(m1, l, r, r2, W));
            const T h = T(0.5);
            return V3{double(h * (l.x + r.x)), double(h * (l.y + r.y)), double(h * (l.z + r.z))};
        };
        V3 cv, G[3], vb = Z;
        const double w = A.bscale * (9.81 * 0.5) / A.tRef;
        double rb[3] = {0, 0, 0};
        if (A.tbar && cell) { const int gi = 3 * g.G(t, j, i); rb[0] = A.rbar[gi]; rb[1] = A.rbar[gi + 1]; rb[2] = A.rbar[gi + 2]; }
        V3 T0 = tk;                                    // to rows j+1 (+) and j-1 (-), plane t
        double h = hk, hj = 0.0;
        // ---- i face ---------------------------------------------------------------------------------
        {
            const T W = okI ? V.x : T(0);            // (what a face that is not evaluated here holds stays out)
            const V3 fc = ld3(A.icsi, c), fe = ld3(A.ieta, c), fz = ld3(A.izet, c);
            const V3 d[3] = {diff(ui, u), four(uji, uj, shdn3(ujm), ujm), four(uki, uk, shdn3(ukm), ukm)};
            const double nuEff = A.les ? A.nu + 0.5 * (double(n0) + double(ni)) : A.nu;
            const V3 F = sel(okI, add3v(fb, sc3(-1.0, fbi)));
            vb.x = opaque_value(okI ? -dot3(F, face_u(uim, u, ui, uii, W)) : 0.0);
            const double nb = adj(std::integral_constant<int, 0>(), okI, F, double(W), d, nuEff, fc, fe, fz, A.iaj[c], cv, G);
            if (face && okI) A.nueb[0][c] = P(nb);
            const bool pos = W > T(0);
            const double wl = QUICK ? (pos ? 0.75 : 0.375) : 0.5, wr = QUICK ? (pos ? 0.375 : 0.75) : 0.5;
            V3 r = add3v(sc3(wr, cv), G[0]);
            if constexpr (QUICK) {
                r = add3v(r, up(sel(!pos, sc3(-0.125, cv))));
                a1 = add3v(a1, dn(sel(pos, sc3(-0.125, cv))));
            }
            a1 = add3v(a1, add3v(add3v(sc3(wl, cv), sc3(-1.0, G[0])), up(r)));
            T0 = add3v(T0, sc3(0.25, add3v(G[1], up(G[1]))));
            const V3 b = sc3(0.25, add3v(G[2], up(G[2])));
            a2 = add3v(a2, b);
            a0 = add3v(a0, sc3(-1.0, b));
            const double hi = cell ? w * fc.z * rb[0] : 0.0;
            h += hi + shup(hi);
        }
        V3 JM = Z;
        // ---- j face ---------------------------------------------------------------------------------
        {
            const T W = okJ ? V.y : T(0);            // (what a face that is not evaluated holds stays out)
            const V3 fc = ld3(A.jcsi, c), fe = ld3(A.jeta, c), fz = ld3(A.jzet, c);
            const V3 d[3] = {four(uji, ui, shup3(uj), uim), diff(uj, u),
                             four(ld3(A.ucat, c + SK + SJ), uk, ld3(A.ucat, c - SK + SJ), ukm)};
            const double nuEff = A.les ? A.nu + 0.5 * (double(n0) + double(nj)) : A.nu;
            const V3 F = sel(okJ, add3v(fb, sc3(-1.0, fbj)));
            Vec3<T> ujj = uj;
            if constexpr (QUICK) ujj = ld3(A.ucat, c + 2 * SJ);
            vb.y = opaque_value(okJ ? -dot3(F, face_u(ujm, u, uj, ujj, W)) : 0.0);
            const double nb = adj(std::integral_constant<int, 1>(), okJ, F, double(W), d, nuEff, fc, fe, fz, A.jaj[c], cv, G);
            if (face && okJ) A.nueb[1][c] = P(nb);
            const bool pos = W > T(0);
            const double wl = QUICK ? (pos ? 0.75 : 0.375) : 0.5, wr = QUICK ? (pos ? 0.375 : 0.75) : 0.5;
            const V3 ld = sc3(0.25, add3v(up(G[0]), sc3(-1.0, dn(G[0]))));
            a1 = add3v(a1, add3v(add3v(sc3(wl, cv), sc3(-1.0, G[1])), ld));
            p1 = add3v(p1, add3v(add3v(sc3(wr, cv), G[1]), ld));
            if constexpr (QUICK) {
                // (selected before the weights: behind them it took the FP64 instance from 10 spilled registers to 18)
                const V3 cl = sel(pos, cv), cr = sel(!pos, cv);
                JM = sc3(pos ? -0.125 : 0.0, cl);
                const V3 q = sc3(-0.125, cr);
                put(sQ[slot], q);
                if (face && (r >= VM_NR - 2 || j >= g.my - 3)) stp3(jpp, c, q);
            }
            const V3 b = sc3(0.25, G[2]);
            a2 = add3v(a2, b);
            a0 = add3v(a0, sc3(-1.0, b));
            p2 = add3v(p2, b);
            p0 = add3v(p0, sc3(-1.0, b));
            hj = cell ? w * fe.z * rb[1] : 0.0;
            h += hj;
        }
        // ---- k face ---------------------------------------------------------------------------------
        {
            const T W = okK ? V.z : T(0);            // (what a face that is not evaluated holds stays out)
            const V3 fc = ld3(A.kcsi, c), fe = ld3(A.keta, c), fz = ld3(A.kzet, c);
            const V3 d[3] = {four(uki, ui, shup3(uk), uim),
                             four(ld3(A.ucat, c + SK + SJ), uj, ld3(A.ucat, c + SK - SJ), ujm), diff(uk, u)};
            const double nuEff = A.les ? A.nu + 0.5 * (double(n0) + double(nk)) : A.nu;
            const V3 F = sel(okK, add3v(fb, sc3(-1.0, fbk)));
            Vec3<T> ukk = uk;
            if constexpr (QUICK) ukk = ld3(A.ucat, c + 2 * SK);
            vb.z = opaque_value(okK ? -dot3(F, face_u(ukm, u, uk, ukk, W)) : 0.0);
            const double nb = adj(std::integral_constant<int, 2>(), okK, F, double(W), d, nuEff, fc, fe, fz, A.kaj[c], cv, G);
            if (face && okK) A.nueb[2][c] = P(nb);
            const bool pos = W > T(0);
            const double wl = QUICK ? (pos ? 0.75 : 0.375) : 0.5, wr = QUICK ? (pos ? 0.375 : 0.75) : 0.5;
            const V3 ld = sc3(0.25, add3v(up(G[0]), sc3(-1.0, dn(G[0]))));
            a1 = add3v(a1, add3v(add3v(sc3(wl, cv), sc3(-1.0, G[2])), ld));
            a2 = add3v(a2, add3v(add3v(sc3(wr, cv), G[2]), ld));
            if constexpr (QUICK) {
                a0 = add3v(a0, sel(pos, sc3(-0.125, cv)));
                a3 = sel(!pos, sc3(-0.125, cv));
            }
            tk = sc3(0.25, G[1]);
            T0 = add3v(T0, tk);
            hk = cell ? w * fz.z * rb[2] : 0.0;
            h += hk;
        }
        p1 = add3v(p1, T0);
        JM = add3v(JM, sc3(-1.0, T0));
        // ---- plane t's jm and theta sums and plane t-1's own and jp sums are complete -----------------
        if (face) {
            if (okI && okJ && okK) stp3(A.vbar, c, vb);
            else {                                     // (the others are the boundary threads' or zero)
                if (okI) A.vbar[3 * c] = T(vb.x);
                if (okJ) A.vbar[3 * c + 1] = T(vb.y);
                if (okK) A.vbar[3 * c + 2] = T(vb.z);
            }
            if (r == 0) stp3(jm, c, JM);
            if (A.tbar) { A.tb[c] = h; A.tb[c + n] = hj; }
        }
        put(sM[slot], JM);
        put(sP[t & 1], p0);
        __syncthreads();
        V3 S = a0;
        if (r >= 1) S = add3v(S, from(sP[t & 1], r - 1));
        if (r < VM_NR - 1) S = add3v(S, from(sM[last], r + 1));
        if constexpr (QUICK) { if (r >= 2) S = add3v(S, from(sQ[last], r - 2)); }
        if (t - 1 >= kb && t - 1 < ke && mine) {
            const int cm = opaque_index(c0 + (t - 1) * SK);
            stp3(own, cm, S);
            if (r == VM_NR - 1 || j == g.my - 2) stp3(jp, cm, p0);
        }
        last = slot;
        slot = slot == 2 ? 0 : slot + 1;
        a0 = a1; a1 = a2; a2 = a3; a3 = Z;
        p0 = p1; p1 = p2; p2 = Z;
    }
}

namespace {
// ucat_bar of point (i, j, k) from the boundary faces' scatter (which only reaches indices up to 2 from
// either side) and the row sums of k_vjp_march: the row's own and, from rows of another workgroup, row j-1's
// jp, row j+1's jm, row j-2's jpp
template <class T, class P>
__device__ __forceinline__ V3 row_sums(const VjpArgs<T, P> &A, const Geo &g, int i, int j, int k, int c) {
    const long n = A.n;
    const int SJ = g.gxm, jl = g.my - 2;
    auto get = [&](int q, int p) { return ldp3(A.rows + 3 * q * n, p); };
    V3 s{0, 0, 0};
    if (i <= 2 || i >= g.mx - 3 || j <= 2 || j >= g.my - 3 || k <= 2 || k >= g.mz - 3) s = cvt3<double>(ld3(A.ubar, c));
    const int r = (j - 1) % VM_NR;                     // (of row 0: -1)
    if (j >= 1 && j <= jl) s = add3v(s, get(0, c));
    if (j >= 2 && j <= jl + 1 && (r == 0 || j == jl + 1)) s = add3v(s, get(1, c - SJ));
    if (j <= jl - 1 && (r == VM_NR - 1 || j == 0)) s = add3v(s, get(2, c + SJ));
    if (A.quick && j >= 3 && j <= jl + 1 && (r <= 1 || j == jl + 1)) s = add3v(s, get(3, c - 2 * SJ));
    return s;
}
// theta_bar of the point: the row's own part and row j-1's j face
template <class T, class P>
__device__ __forceinline__ T theta_sum(const VjpArgs<T, P> &A, const Geo &g, int j, int c) {
    double s = 0.0;
    if (j >= 1 && j <= g.my - 2) s = A.tb[c];
    if (j >= 2 && j <= g.my - 1) s += A.tb[A.n + c - g.gxm];
    return T(s);
}
// nu_t_bar of an interior cell is half the nu_eff cotangents of its six faces and of the boundary faces
// whose ghost nu_t UpdateNutBCs fills from this cell.  Along one axis (x of 1 .. m-2, point stride st) that
// is hi times the face at the cell's own index and lo times the face `off` points from it: the one below,
// or the last face for the first cell of a periodic axis, whose face 0 is not evaluated
struct NuFaces { double hi, lo; int off; };
template <class A_>
__device__ __forceinline__ NuFaces nu_faces(const A_ &A, const Geo &g, int q, int x, int st) {
    const int m = q == 0 ? g.mx : q == 1 ? g.my : g.mz;
    const int bl = A.bc_nut[2 * q], br = A.bc_nut[2 * q + 1];
    NuFaces f{x == m - 2 && br == TOSCA_BCNUT_ZEROGRADIENT ? 2.0 : 1.0, 1.0, -st};
    if (x == 1 && g.per[q] == TOSCA_PERIODIC_NONE) f.lo = bl == TOSCA_BCNUT_ZEROGRADIENT ? 2.0 : 1.0;
    else if (x == 1) { f.lo = br == TOSCA_BCNUT_PERIODIC ? 1.0 : 0.0; f.off = br == TOSCA_BCNUT_PERIODIC ? (m - 3) * st : -st; }
    return f;
}
// du_center of a cell at index x of an axis, transposed: what its derivative cotangent adds to the cell
// above, the cell below and the cell itself (one-sided at the first and last cell of a non-periodic axis)
__device__ __forceinline__ double w_up(bool np, int x, int m) { return np && x == m - 2 ? 0.0 : np && x == 1 ? 1.0 : 0.5; }
__device__ __forceinline__ double w_dn(bool np, int x, int m) { return np && x == m - 2 ? -1.0 : np && x == 1 ? 0.0 : -0.5; }
__device__ __forceinline__ double w_own(bool np, int x, int m) { return np && x == m - 2 ? 1.0 : np && x == 1 ? -1.0 : 0.0; }
// such a weight times v; a weight of zero takes nothing, also of a v that is not finite
__device__ __forceinline__ V3 wt3(double w, V3 v) { return V3{w != 0.0 ? w * v.x : 0.0, w != 0.0 ? w * v.y : 0.0, w != 0.0 ? w * v.z : 0.0}; }
}  // namespace

// ------------------------------------------------------------------------------------------------
// ucat_bar and theta_bar of every owned point with nu_t = Cs Delta^2 |S| recomputed: the row sums, and the
// |S| path of the interior cells (nu_t_bar, Cs_bar, the cotangents of the three du_center vectors), which
// a workgroup of 8 rows marching along k keeps on chip: along i by lane shifts, along j through LDS (one
// barrier a plane), along k in the accumulators of three planes.  62 x 6 points a workgroup.
// Bound by memory and by the latency of its loads: 240 bytes a point in FP64, 368 moved at 4.5 TB/s; 0.38 ms on the
// 192 x 192 x 128 hill, 0.54 on the mixed 384 x 256 x 96 box.  Every load of a cell is issued without a branch (with every row's sums read, the
// six faces of nu_t_bar with a condition each took 0.49 and 0.86, 0.43 and 0.62 without); loading the row sums
// ahead of the barrier as well cost 169 registers for 128 and with them half the waves: 0.50 ms.  The launch
// bound holds it at 128 (132 of the compiler's own choice would leave three waves a SIMD).
// ------------------------------------------------------------------------------------------------
constexpr int VF_NR = 8, VF_TI = 62, VF_TJ = VF_NR - 2;
template <class T, class P>
__global__ void __launch_bounds__(64 * VF_NR, 4) k_vjp_finish(VjpArgs<T, P> A, Geo g, int kchunk) {
    __shared__ double sG[2][3][VF_NR][64];
    const int lane = threadIdx.x, r = threadIdx.y;
    const int tile = xcd_tile();                       // j fastest, then i, then the k chunk
    const int bj = tile % gridDim.y, bi = (tile / gridDim.y) % gridDim.x, bk = tile / (gridDim.x * gridDim.y);
    const int i = bi * VF_TI + lane - 1, j = bj * VF_TJ + r - 1;
    const int kb = bk * kchunk, ke = min(kb + kchunk, g.mz);     // points [kb, ke)
    const bool mine = lane >= 1 && lane <= VF_TI && r >= 1 && r <= VF_TJ && i < g.mx && j < g.my;
    const bool cellIJ = i >= 1 && i <= g.mx - 2 && j >= 1 && j <= g.my - 2;
    const bool np0 = g.nonper(0), np1 = g.nonper(1), np2 = g.nonper(2);
    const double wuI = w_up(np0, i, g.mx), wdI = w_dn(np0, i, g.mx), woI = w_own(np0, i, g.mx), woJ = w_own(np1, j, g.my);
    const double wuJ = w_up(np1, j - 1, g.my), wdJ = w_dn(np1, j + 1, g.my);     // of the rows below and above
    const int rm = max(r - 1, 0), rp = min(r + 1, VF_NR - 1);
    const int SJ = g.gxm, SK = g.gxm * g.gym;
    const int p0 = g.L(0, min(j, g.my), min(i, g.mx));           // the point in plane 0 (indices from -1)
    const NuFaces fi = nu_faces(A, g, 0, i, 1), fj = nu_faces(A, g, 1, j, SJ);
    V3 c0{0, 0, 0}, c1{0, 0, 0}, c2{0, 0, 0};          // sums of the points of planes k-1, k, k+1
    Vec3<T> um = ld3(A.ucat, p0 + (kb - 2) * SK), u = ld3(A.ucat, p0 + (kb - 1) * SK);
    for (int k = kb - 1; k <= ke; k++) {
        const int buf = k & 1;
        const bool cell = cellIJ && k >= 1 && k <= g.mz - 2;
        // every load of the plane without a branch, so that they are in flight together
        const int c = opaque_index(p0 + k * SK);
        const NuFaces fk = nu_faces(A, g, 2, k, SK);
        const double nb = 0.5 * (fi.hi * double(A.nueb[0][c]) + fi.lo * double(A.nueb[0][c + fi.off]) +
                                 fj.hi * double(A.nueb[1][c]) + fj.lo * double(A.nueb[1][c + fj.off]) +
                                 fk.hi * double(A.nueb[2][c]) + fk.lo * double(A.nueb[2][c + fk.off]));
        const V3 cc = ld3(A.csi, c), ee = ld3(A.eta, c), zz = ld3(A.zet, c);
        const double a = A.aj[c], cs = A.cs[c];
        const Vec3<T> up = ld3(A.ucat, c + SK);
        const GradT<T> gr = du_center_v(g, i, j, k, u, ld3(A.ucat, c - 1), ld3(A.ucat, c + 1), ld3(A.ucat, c - SJ),
                                        ld3(A.ucat, c + SJ), um, up);
        um = u;
        u = up;
        // the strain as the forward computes it (in T), the rest in FP64
        const CartT<T> dT = du_dxyz(cvt3<T>(cc), cvt3<T>(ee), cvt3<T>(zz), T(a), gr);
        const double S = double(strain_mag(dT));
        const double filter = cube_root(1. / a), d2 = filter * filter;
        if (cell && mine && k >= kb && k < ke) A.csbar[c] = nb * d2 * S;
        // d|S| / dD_mn = 2 S_mn / |S|, S = sym(D); |S| is not differentiable at 0: subgradient 0
        const bool on = cell && S != 0.0 && nb != 0.0;
        const double sb = nb * cs * d2 * 2.0 / S;
        const double Sxx = dT.du_dx, Sxy = 0.5 * (double(dT.du_dy) + double(dT.dv_dx)), Sxz = 0.5 * (double(dT.du_dz) + double(dT.dw_dx));
        const double Syy = dT.dv_dy, Syz = 0.5 * (double(dT.dv_dz) + double(dT.dw_dy)), Szz = dT.dw_dz;
        const V3 Du{sb * Sxx, sb * Sxy, sb * Sxz}, Dv{sb * Sxy, sb * Syy, sb * Syz}, Dw{sb * Sxz, sb * Syz, sb * Szz};
        // D_m. = aj (d_c u_m csi + d_e u_m eta + d_z u_m zet)  ->  d_X u_m bar = aj (Dbar_m . M_X)
        auto bar = [&](V3 M) {
            const V3 v{a * dot3(Du, M), a * dot3(Dv, M), a * dot3(Dw, M)};
            return V3{on ? v.x : 0.0, on ? v.y : 0.0, on ? v.z : 0.0};
        };
        const V3 gc = bar(cc), ge = bar(ee), gz = bar(zz);
        sG[buf][0][r][lane] = ge.x; sG[buf][1][r][lane] = ge.y; sG[buf][2][r][lane] = ge.z;
        // own cell, then the cells along i
        const double woK = w_own(np2, k, g.mz);
        c1 = add3v(c1, add3v(wt3(woI, gc), add3v(wt3(woJ, ge), wt3(woK, gz))));
        c1 = add3v(c1, add3v(shup3(wt3(wuI, gc)), shdn3(wt3(wdI, gc))));
        c2 = add3v(c2, wt3(w_up(np2, k, g.mz), gz));
        c0 = add3v(c0, wt3(w_dn(np2, k, g.mz), gz));
        __syncthreads();                               // the other buffer is rewritten behind the next one
        c1 = add3v(c1, add3v(wt3(wuJ, V3{sG[buf][0][rm][lane], sG[buf][1][rm][lane], sG[buf][2][rm][lane]}),
                             wt3(wdJ, V3{sG[buf][0][rp][lane], sG[buf][1][rp][lane], sG[buf][2][rp][lane]})));
        if (mine && k - 1 >= kb && k - 1 < ke) {       // the points of plane k-1 are complete
            const int cm = opaque_index(p0 + (k - 1) * SK);
            stp3(A.ubar, cm, add3v(row_sums(A, g, i, j, k - 1, cm), c0));
            if (A.tbar) A.tbar[cm] = theta_sum(A, g, j, cm);
        }
        c0 = c1; c1 = c2; c2 = V3{0, 0, 0};
    }
}

// ------------------------------------------------------------------------------------------------
// The same without the |S| path (no LES, or nu_t an input array): one thread per owned point.  With nu_t
// an input its cotangent is accumulated (+=): the face of direction q at index point c averages nu_t of
// cells c and c + e_q, so point c collects half the nu_eff cotangent of faces c and c - e_q (zero where a
// face is not evaluated).
// ------------------------------------------------------------------------------------------------
template <class T, class P>
__global__ void __launch_bounds__(256) k_vjp_sum(VjpArgs<T, P> A, Geo g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
    if (i > g.mx - 1 || j > g.my - 1) return;
    const int c = g.L(k, j, i);
    stp3(A.ubar, c, row_sums(A, g, i, j, k, c));
    if (A.tbar) A.tbar[c] = theta_sum(A, g, j, c);
    if (A.les && A.nutbar_acc) {
        const double s = double(A.nueb[0][c]) + double(A.nueb[0][g.L(k, j, i - 1)]) + double(A.nueb[1][c]) +
                         double(A.nueb[1][g.L(k, j - 1, i)]) + double(A.nueb[2][c]) + double(A.nueb[2][g.L(k - 1, j, i)]);
        A.nutbar_acc[c] += 0.5 * s;
    }
}

// The transposed stages on the stream.  cs != nullptr: nu_t = UpdateNut(ucat, cs) is recomputed
// and differentiated (Cs_bar, |S| path); nut_in != nullptr: nu_t is an input and its cotangent is
// added to nut_bar.  theta_bar == nullptr: no Buoyancy term.  ws (vjp_ws_doubles): n values of T for
// nu_t, 2 n doubles for tb, then 18 n values of P for fpbar, nueb and the row sums.
template <class T, class P>
void vjp_rhs_impl(const Geo &g, const tosca_mesh *mesh, const tosca_params *p, const T *ucont, const T *ucat,
                  const double *cs, const T *nut_in, const double *rbar, double scale, double buoy_scale, T *ucont_bar,
                  T *ucat_bar, T *theta_bar, double *cs_bar, double *nut_bar, double *ws, hipStream_t s) {
    const long n = g.nloc();
    T *nut = reinterpret_cast<T *>(ws);
    P *base = reinterpret_cast<P *>(ws + 3 * n);
    P *fpbar = base, *nueb = base + 3 * n;
    const bool les = p->les_active != 0;
    const bool renut = les && !nut_in;      // nu_t recomputed as the forward step does (k_vjp_pre)
    // what no later kernel writes: ucont_bar, nueb and cs_bar outside the interior cells (k_vjp_march writes
    // every face of theirs), theta_bar outside the owned points; and the layers of
    // ucat_bar the boundary faces scatter into
    ZeroShells Z{};
    auto zero = [&](void *p, int words, int w) { if (p) { Z.p[Z.n] = static_cast<unsigned *>(p); Z.words[Z.n] = words; Z.w[Z.n++] = w; } };
    const int wT = sizeof(T) / 4, wP = sizeof(P) / 4;
    zero(ucont_bar, 3 * wT, GW + 1);
    zero(ucat_bar, 3 * wT, GW + 3);
    zero(theta_bar, wT, GW);
    zero(cs_bar, 2, renut ? GW + 1 : g.gzm);           // (without the |S| path, all of it)
    for (int q = 0; q < 3; q++) zero(nueb + q * n, wP, GW + 1);
    TOSCA_LAUNCH("k_vjp_zero", k_vjp_zero_shells, dim3(256, 6, Z.n), dim3(256), 0, s, Z, g);
    VjpArgs<T, P> A;
    A.ucont = ucont; A.ucat = ucat; A.cs = cs; A.rbar = rbar;
    A.nut = les ? (nut_in ? nut_in : nut) : ucat;
    A.nut_w = nut;
    A.csi = mesh->csi; A.eta = mesh->eta; A.zet = mesh->zet;
    A.icsi = mesh->icsi; A.ieta = mesh->ieta; A.izet = mesh->izet;
    A.jcsi = mesh->jcsi; A.jeta = mesh->jeta; A.jzet = mesh->jzet;
    A.kcsi = mesh->kcsi; A.keta = mesh->keta; A.kzet = mesh->kzet;
    A.aj = mesh->aj; A.iaj = mesh->iaj; A.jaj = mesh->jaj; A.kaj = mesh->kaj;
    A.fpbar = fpbar; A.nutbar_acc = nut_bar;
    A.vbar = ucont_bar; A.ubar = ucat_bar; A.tbar = theta_bar; A.csbar = cs_bar;
    for (int q = 0; q < 3; q++) A.nueb[q] = nueb + q * n;
    A.rows = base + 6 * n;
    A.tb = ws + n;
    A.n = n;
    A.scale = scale; A.bscale = buoy_scale; A.tRef = p->t_ref; A.nu = p->nu;
    A.quick = p->div_scheme == TOSCA_DIV_QUICK;
    A.les = les;
    for (int q = 0; q < 6; q++) { A.bc_u[q] = p->bc_u[q]; A.bc_nut[q] = p->bc_nut[q]; }
    const bool f32 = sizeof(T) == 4;
    const dim3 cb(64, 4), cg((g.mx - 2 + 63) / 64, (g.my - 2 + 3) / 4, g.mz - 2);
    if (renut) {
        TOSCA_LAUNCH(f32 ? "k_vjp_pre_f32" : "k_vjp_pre", (k_vjp_pre<T, P>), cg, cb, 0, s, A, g);
        launch_nut_ghosts(nut, p, g, s);
    } else {
        TOSCA_LAUNCH(f32 ? "k_vjp_fp_f32" : "k_vjp_fp", (k_vjp_fp<T, P>), cg, cb, 0, s, A, g);
    }
    const int ti = (g.mx + 59) / 60, tj = (g.my - 2 + VM_NR - 1) / VM_NR;
    const int kc = plane_chunk(g.mz, ti * tj, CHUNK_VJP_MARCH);
    const int nmax = max(g.my * g.mz, max(g.mx * g.mz, g.mx * g.my));
    const int nbnd = (6 * nmax + 64 * VM_NR * NUM_XCD - 1) / (64 * VM_NR * NUM_XCD) * NUM_XCD;     // a multiple of the XCDs
    const dim3 mg(nbnd + ti * tj * ((g.mz + kc - 1) / kc));
    if (A.quick) TOSCA_LAUNCH(f32 ? "k_vjp_march_f32" : "k_vjp_march", (k_vjp_march<T, P, true>), mg, dim3(64, VM_NR), 0, s, A, g, kc, ti, tj, nbnd, nmax);
    else TOSCA_LAUNCH(f32 ? "k_vjp_march_f32" : "k_vjp_march", (k_vjp_march<T, P, false>), mg, dim3(64, VM_NR), 0, s, A, g, kc, ti, tj, nbnd, nmax);
    if (renut) {
        const int fi = (g.mx + VF_TI - 1) / VF_TI, fj = (g.my + VF_TJ - 1) / VF_TJ;
        const int fc = plane_chunk(g.mz, fi * fj, CHUNK_VJP_FINISH);
        TOSCA_LAUNCH(f32 ? "k_vjp_finish_f32" : "k_vjp_finish", (k_vjp_finish<T, P>), dim3(fi, fj, (g.mz + fc - 1) / fc),
                     dim3(64, VF_NR), 0, s, A, g, fc);
    } else {
        TOSCA_LAUNCH(f32 ? "k_vjp_sum_f32" : "k_vjp_sum", (k_vjp_sum<T, P>), dim3((g.mx + 63) / 64, (g.my + 3) / 4, g.mz),
                     dim3(64, 4), 0, s, A, g);
    }
}

size_t vjp_ws_doubles(const Geo &g) { return 21 * (size_t)g.nloc(); }

void vjp_rhs(const Geo &g, const tosca_mesh *mesh, const tosca_params *p, const double *ucont, const double *ucat,
             const double *theta, const double *cs, const double *rbar, double scale, double buoy_scale,
             double *ucont_bar, double *ucat_bar, double *theta_bar, double *cs_bar, double *ws, hipStream_t s) {
    vjp_rhs_impl<double, double>(g, mesh, p, ucont, ucat, cs, nullptr, rbar, scale, buoy_scale, ucont_bar, ucat_bar,
                                 theta_bar, cs_bar, nullptr, ws, s);
}

void vjp_rhs_mixed(const Geo &g, const tosca_mesh *mesh, const tosca_params *p, const float *ucont, const float *ucat,
                   const double *cs, const double *rbar, double scale, double buoy_scale, float *ucont_bar,
                   float *ucat_bar, float *theta_bar, double *cs_bar, double *ws, hipStream_t s) {
    vjp_rhs_impl<float, float>(g, mesh, p, ucont, ucat, cs, nullptr, rbar, scale, buoy_scale, ucont_bar, ucat_bar,
                               theta_bar, cs_bar, nullptr, ws, s);
}

// FormU(formMode 0, scale) as a function of (ucont, ucat, nu_t): ucont_bar and ucat_bar
// overwritten, the nu_t cotangent added to nut_bar (when LES is active)
void vjp_formu_nut(const Geo &g, const tosca_mesh *mesh, const tosca_params *p, const double *ucont, const double *ucat,
                   const double *nut, const double *rbar, double scale, double *ucont_bar, double *ucat_bar,
                   double *nut_bar, double *ws, hipStream_t s) {
    vjp_rhs_impl<double, double>(g, mesh, p, ucont, ucat, nullptr, p->les_active ? nut : nullptr, rbar, scale, 0.0,
                                 ucont_bar, ucat_bar, nullptr, nullptr, nut_bar, ws, s);
}

}  // namespace tosca
