// harm_eos5d.hpp -- tabulated equation of state and the 5D primitive
// solver (utoprim_5d.c) for the gfx950 kernels (FP64).
//
// The table holds e(rho, T) and p(rho, T) on an increasing (rho, T) grid in
// code units.  p(rho, u) is the piecewise-bilinear interpolant in (rho, T),
// inverted along T at fixed rho by bisection over the cell edges and one exact
// linear solve inside the cell: no transcendental function, so the CPU oracle
// evaluates the same numbers bit for bit.  Outside the table the Gamma-law
// pressure is used, as the reference does outside its table
// (cooleos.c:342-366).  The reference evaluates p(rho, u) by a T-Newton on an
// Akima spline of its cached table (cooleos.c:314-444) and keeps the last T
// per zone as the next start; the direct inversion here needs no such state.
#pragma once
#include <hip/hip_runtime.h>

namespace harm {

struct EosTab {
    int nr, nt;
    const double *rho, *T, *e, *p;  // device, rho[nr], T[nt], e/p [nr][nt]
    double gam;                     // Gamma-law fallback outside the table
};

__device__ __forceinline__ int eos_cell(const double *x, int n, double v)
{
    int lo = 0, hi = n - 1;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (x[mid] <= v)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// p(rho, u), dp/drho at fixed u, dp/du at fixed rho; 1 on the Gamma-law branch.
// T (optional) receives the temperature along the same interpolation, 0 on the
// Gamma-law branch.
__device__ inline int eos_table_p(const EosTab &t, double rho, double u, double &p, double &dpdrho, double &dpdu,
                                  double *T = nullptr)
{
    const int nr = t.nr, nt = t.nt;
    if (rho >= t.rho[0] && rho <= t.rho[nr - 1]) {
        const int k = eos_cell(t.rho, nr, rho);
        const double dr = t.rho[k + 1] - t.rho[k];
        const double a = (rho - t.rho[k]) / dr;
        const double *e0 = t.e + (size_t)k * nt, *e1 = e0 + nt;
        const double *p0 = t.p + (size_t)k * nt, *p1 = p0 + nt;
        auto EAT = [&](int j) { return e0[j] + a * (e1[j] - e0[j]); };
        const double Elo = EAT(0), Ehi = EAT(nt - 1);
        if (u >= Elo && u <= Ehi) {
            int lo = 0, hi = nt - 1;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (EAT(mid) <= u)
                    lo = mid;
                else
                    hi = mid;
            }
            const double E0 = EAT(lo), E1 = EAT(lo + 1);
            const double P0 = p0[lo] + a * (p1[lo] - p0[lo]);
            const double P1 = p0[lo + 1] + a * (p1[lo + 1] - p0[lo + 1]);
            const double dE = E1 - E0, dP = P1 - P0;
            const double b = (u - E0) / dE;
            p = P0 + b * dP;
            dpdu = dP / dE;
            const double sE0 = (e1[lo] - e0[lo]) / dr, sE1 = (e1[lo + 1] - e0[lo + 1]) / dr;
            const double sP0 = (p1[lo] - p0[lo]) / dr, sP1 = (p1[lo + 1] - p0[lo + 1]) / dr;
            dpdrho = sP0 + (-sE0 * dP * dE + (u - E0) * ((sP1 - sP0) * dE - dP * (sE1 - sE0))) / (dE * dE);
            if (T) *T = t.T[lo] + b * (t.T[lo + 1] - t.T[lo]);
            return 0;
        }
    }
    p = (t.gam - 1.) * u;
    dpdrho = 0.;
    dpdu = t.gam - 1.;
    if (T) *T = 0.;
    return 1;
}

// The 5D solver's view of the EOS: tab == nullptr is the Gamma-law pressure.  at() is
// called once per iterate: its pressure serves the residual, the Jacobian and the
// step's W, where each searched the table again (three times an iterate).
struct Eos5 {
    const EosTab *tab;
    double gam;
    __device__ bool tabulated() const { return tab != nullptr; }
    __device__ EosPt at(double rho, double u) const
    {
        EosPt e{(gam - 1.) * u, 0., 0.};
        if (tab) eos_table_p(*tab, rho, u, e.p, e.dpdrho, e.dpdu);
        return e;
    }
    __device__ void derivs(double, double, EosPt &) const {}
    __device__ void refresh(Geom &) const {}
};

// ---- utoprim_5d.c, restated for one zone -----------------------------------
constexpr int N5 = 5;

// The numbers of one zone's metric and field that every iterate uses.
struct Zone5 {
    double lapse;          // sqrt(-1 / g^tt) (ncov_calc, u2p_util.c:204-210; n_t = -lapse)
    double alpha, ralpha;  // 1 / sqrt(-g^tt) (u2p_util.c:95) and its reciprocal
    double boa[4];         // beta^j / alpha, beta^j = g^tj alpha alpha
};

__device__ __forceinline__ Zone5 zone5(const Geom &g)
{
    Zone5 z;
    z.lapse = sqrt(-1. / g.gcon[0][0]);
    z.alpha = 1.0 / sqrt(-g.gcon[0][0]);
    z.ralpha = 1.0 / z.alpha;
    z.boa[0] = 0.;
#pragma unroll
    for (int j = 1; j < 4; j++) z.boa[j] = g.gcon[0][j] * z.alpha * z.alpha / z.alpha;
    return z;
}

__device__ __forceinline__ void lower_g5(const double *vcon, const Geom &g, double *vcov)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        vcov[i] = g.gcov[i][0] * vcon[0];
#pragma unroll
        for (int j = 1; j < 4; j++) vcov[i] += g.gcov[i][j] * vcon[j];
    }
}

// gamma_calc_g (u2p_util.c:319-341); on failure gamma = sqrt(1 + |utsq|).
__device__ __forceinline__ int gamma_calc_g5(const double *pr, const Geom &g, double &gamma)
{
    double utsq = g.gcov[1][1] * pr[U1] * pr[U1] + g.gcov[2][2] * pr[U2] * pr[U2] + g.gcov[3][3] * pr[U3] * pr[U3] +
                  2. * (g.gcov[1][2] * pr[U1] * pr[U2] + g.gcov[1][3] * pr[U1] * pr[U3] +
                        g.gcov[2][3] * pr[U2] * pr[U3]);
    int bad = 0;
    if (utsq < 0.0) {
        if (fabs(utsq) > 1.E-10) bad = 1;
        utsq = fabs(utsq);
    }
    gamma = fsqrt(1. + utsq);
    return bad;
}

// The linear solve of one Newton step (LU_decompose / LU_substitution,
// utoprim_5d.c:672-874), B its right-hand side and result.  The row swaps act on B as
// on A's columns: the reference swaps B during the forward substitution, at step i only
// among rows i and below, which that substitution has not reached.
__device__ inline void lu5_solve(double (&A)[N5][N5], double (&B)[N5])
{
    const double absmin = 1e-30;
    double row_norm[N5];
    const int n = N5;
    bool zero = false;
#pragma unroll
    for (int i = 0; i < n; i++) {
        double absmax = 0.;
#pragma unroll
        for (int j = 0; j < n; j++) absmax = fmax(absmax, fabs(A[i][j]));
        zero |= absmax == 0.;
        row_norm[i] = fdiv(1., absmax);
    }
    if (zero) {
        // the reference returns before factorizing and then substitutes with the
        // unfactorized matrix and a zero permutation
#pragma unroll
        for (int i = 0; i < n; i++) {
            double tmpvar = B[0];
            B[0] = B[i];
#pragma unroll
            for (int j = i - 1; j >= 0; j--) tmpvar -= A[i][j] * B[j];
            B[i] = tmpvar;
        }
    } else {
#pragma unroll
        for (int j = 0; j < n; j++) {
#pragma unroll
            for (int i = 0; i < j; i++)
#pragma unroll
                for (int k = 0; k < i; k++) A[i][j] -= A[i][k] * A[k][j];
            double absmax = 0.0;
            int max_row = j;
#pragma unroll
            for (int i = j; i < n; i++) {
#pragma unroll
                for (int k = 0; k < j; k++) A[i][j] -= A[i][k] * A[k][j];
                const double m = fabs(A[i][j]) * row_norm[i];
                if (m >= absmax) {
                    absmax = m;
                    max_row = i;
                }
            }
            if (max_row != j && !((j == (n - 2)) && (A[j][j + 1 < n ? j + 1 : j] == 0.))) {
                // rows j and max_row by selects: the rows are registers
#pragma unroll
                for (int r = j + 1; r < n; r++) {
                    const bool sw = r == max_row;
#pragma unroll
                    for (int k = 0; k < n; k++) {
                        const double a = A[j][k], b = A[r][k];
                        A[j][k] = sw ? b : a;
                        A[r][k] = sw ? a : b;
                    }
                    const double a = B[j], b = B[r];
                    B[j] = sw ? b : a;
                    B[r] = sw ? a : b;
                    row_norm[r] = sw ? row_norm[j] : row_norm[r];
                }
            }
            if (A[j][j] == 0.) A[j][j] = absmin;
            if (j != (n - 1)) {
                const double inv = fdiv(1., A[j][j]);
#pragma unroll
                for (int i = j + 1; i < n; i++) A[i][j] *= inv;
            }
        }
#pragma unroll
        for (int i = 0; i < n; i++)
#pragma unroll
            for (int j = i - 1; j >= 0; j--) B[i] -= A[i][j] * B[j];
    }
#pragma unroll
    for (int i = n - 1; i >= 0; i--) {
#pragma unroll
        for (int j = i + 1; j < n; j++) B[i] -= A[i][j] * B[j];
        B[i] = fdiv(B[i], A[i][i]);
    }
}

// func_5d (utoprim_5d.c:250-359), NORMMETHOD 1, with primtoU_g (u2p_util.c:84-145) and
// dudp_calc_g (utoprim_5d.c:409-529, its helpers 531-640): the Newton step dx, f and df
// at the iterate x with the EOS numbers e.  The two share the four-velocity and the
// field's four-vector; quotients by one denominator (u^t, alpha, u_t, the field's
// gamma) go through its reciprocal (div_r, correctly rounded); the reference's sums
// start from 0 and carry terms with the zero components, which change no value.
template <class E5>
__device__ inline void func_5d(const E5 &eos, const double *U_target, const Geom &g, const Zone5 &z, const double *x,
                               const double *Bf, EosPt e, double (&dx)[N5], double &f, double &df)
{
    double ucon[4], ucov[4], bcon[4], bcov[4], Bcov[4], resid[N5], Am[N5][N5];
    {
        double utsq = 0.;
#pragma unroll
        for (int i = 1; i < 4; i++)
#pragma unroll
            for (int j = 1; j < 4; j++) utsq += g.gcov[i][j] * x[UU + i] * x[UU + j];
        const double gamma = fsqrt(1. + fabs(utsq));
        const double lg = z.lapse * gamma;
        ucon[0] = 0. - lg * g.gcon[0][0];
#pragma unroll
        for (int i = 1; i < 4; i++) ucon[i] = x[UU + i] - lg * g.gcon[0][i];
    }
    lower_g5(ucon, g, ucov);
    const double gb = ucon[0] * z.lapse;
    {
        double Bn[4], u_dot_B = 0.;
        Bn[0] = 0.;
#pragma unroll
        for (int i = 1; i < 4; i++) {
            Bn[i] = z.lapse * Bf[i - 1];
            u_dot_B += ucov[i] * Bn[i];
        }
        const double rgb = fdiv(1., gb);
#pragma unroll
        for (int i = 0; i < 4; i++) bcon[i] = div_r(Bn[i] + ucon[i] * u_dot_B, gb, rgb);
    }
    lower_g5(bcon, g, bcov);
    const double bsq = bcon[0] * bcov[0] + bcon[1] * bcov[1] + bcon[2] * bcov[2] + bcon[3] * bcov[3];
    df = 0.;
    {
        const double w = x[RHO] + x[UU] + e.p;
        const double ndb = -z.lapse * bcon[0];
        double Uc[N5];
        Uc[RHO] = ucon[0] * x[RHO];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            double t = gb * (w + bsq) * ucov[i];
            if (i == 0) t -= (e.p + bsq / 2.) * -z.lapse;
            Uc[1 + i] = div_r(t + ndb * bcov[i], z.alpha, z.ralpha);
        }
        Uc[1] = Uc[1] + Uc[RHO];
#pragma unroll
        for (int k = 0; k < N5; k++) {
            const double u = Uc[k] * g.g;
            resid[k] = u - U_target[k];
            double residnorm = 0.5 * (fabs(u) + fabs(U_target[k]));
            residnorm = (residnorm == 0.) ? 1. : fdiv(1., residnorm);
            df -= residnorm * resid[k] * resid[k];
        }
    }
    f = -0.5 * df;

    const double ru = fdiv(1., ucon[0]), rut = fdiv(1., ucov[0]);
    const double bu = div_r(bcon[0], ucon[0], ru);
    Bcov[0] = 0.;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        Bcov[j] = g.gcov[j][1] * Bf[0];
        Bcov[j] += g.gcov[j][2] * Bf[1];
        Bcov[j] += g.gcov[j][3] * Bf[2];
    }
    if (eos.tabulated()) {
        eos.derivs(x[RHO], x[UU], e);
        Am[RHO][RHO] = ucon[0];
        Am[RHO][UU] = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            Am[UU + j][RHO] = (1.0 + e.dpdrho) * ucon[0] * ucov[j];
            Am[UU + j][UU] = (1.0 + e.dpdu) * ucon[0] * ucov[j];
        }
        Am[UU][RHO] += e.dpdrho;
        Am[UU][UU] += e.dpdu;
    } else {
        const double GAMMA = eos.gam;
        Am[RHO][RHO] = ucon[0];
        Am[RHO][UU] = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            Am[UU + j][RHO] = ucon[0] * ucov[j];
            Am[UU + j][UU] = GAMMA * ucon[0] * ucov[j];
        }
        Am[UU][UU] += GAMMA - 1.0;
    }
    const double eta = eos.tabulated() ? x[RHO] + x[UU] + e.p + bsq : x[RHO] + eos.gam * x[UU] + bsq;
    // dU/du^k
    double At[N5][3];
#pragma unroll
    for (int k = 1; k < 4; k++) {
        const double dut = div_r(-ucov[k], ucov[0], rut);
        const double dbt = Bcov[k] + Bcov[0] * dut;
        double dbi[4], dbsq;
        dbi[0] = dbt;
#pragma unroll
        for (int j = 1; j < 4; j++) {
            dbi[j] = div_r(-bcon[j] * dut, ucon[0], ru) + div_r(ucon[j] * dbt, ucon[0], ru);
            if (j == k) dbi[j] += bu;
        }
        dbsq = 2. * bcov[0] * dbi[0];
#pragma unroll
        for (int j = 1; j < 4; j++) dbsq += 2. * bcov[j] * dbi[j];
        At[RHO][k - 1] = x[RHO] * dut;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double dud = g.gcov[j][k] + g.gcov[j][0] * dut;
            double dbd = g.gcov[j][0] * dbi[0];
#pragma unroll
            for (int l = 1; l < 4; l++) dbd += g.gcov[j][l] * dbi[l];
            double a = dbsq * ucon[0] * ucov[j] + eta * (dut * ucov[j] + ucon[0] * dud);
            if (j == 0) a += 0.5 * dbsq;
            At[UU + j][k - 1] = a - (dbt * bcov[j] + bcon[0] * dbd);
        }
    }
    Am[UU][RHO] += Am[RHO][RHO];
    Am[UU][UU] += Am[RHO][UU];
#pragma unroll
    for (int k = 0; k < 3; k++) At[UU][k] += At[RHO][k];
    // du^l/dv^j, l = 1..3 (the reference's product leaves l = 0 out)
    double dg[4];
    {
        double gamma;
        gamma_calc_g5(x, g, gamma);
        const double ig = fdiv(1.0, gamma);
#pragma unroll
        for (int j = 1; j < 4; j++) {
            dg[j] = ig * g.gcov[j][1] * x[U1];
            dg[j] += ig * g.gcov[j][2] * x[U2];
            dg[j] += ig * g.gcov[j][3] * x[U3];
        }
    }
#pragma unroll
    for (int i = 0; i < N5; i++)
#pragma unroll
        for (int j = 1; j < 4; j++) {
            double a = 0.;
#pragma unroll
            for (int l = 1; l <= 3; l++) {
                const double d = (j == l ? 1. : 0.) - z.boa[l] * dg[j];
                a = l == 1 ? At[i][0] * d : a + At[i][l - 1] * d;
            }
            Am[i][U1 + j - 1] = a * g.g;
        }
#pragma unroll
    for (int i = 0; i < N5; i++) {
        Am[i][RHO] *= g.g;
        Am[i][UU] *= g.g;
    }
    double norm = 0.0;
    int numnormterms = 0;
#pragma unroll
    for (int j = 0; j < N5; j++)
#pragma unroll
        for (int k = 0; k < N5; k++)
            if (Am[j][k] > 2.2204460492503131e-16) {
                norm += fabs(Am[j][k]);
                numnormterms++;
            }
    norm = fdiv((double)(numnormterms), norm);
#pragma unroll
    for (int j = 0; j < N5; j++)
#pragma unroll
        for (int k = 0; k < N5; k++) Am[j][k] *= (norm);
#pragma unroll
    for (int k = 0; k < N5; k++) dx[k] = -resid[k] * (norm);
    lu5_solve(Am, dx);
}

// Utoprim_5d (utoprim_5d.c:179-239) with general_newton_raphson
// (utoprim_5d.c:890-983) and calc_errx_5d (utoprim_5d.c:378-400).
// e: the EOS at prim's density and energy.  E5::refresh may read the metric again, where
// at() needs the registers that would hold it.
template <class E5>
__device__ inline int utoprim_5d(const double *U, Geom &g, const E5 &eos, EosPt e, double *prim, int &n_iter_out)
{
#pragma unroll
    for (int k = B1; k <= B3; k++) prim[k] = U[k] / g.g;
    double x[N5];
#pragma unroll
    for (int k = 0; k < N5; k++) x[k] = prim[k];
    const Zone5 z5 = zone5(g);
    double f = 1., df = 1., errx = 1., W = 0.;
    int n_iter = 0, i_extra = 0, doing_extra = 0;
    bool keep = true;
    while (keep) {
        double dx[N5];
        eos.refresh(g);
        func_5d(eos, U, g, z5, x, prim + B1, e, dx, f, df);
#pragma unroll
        for (int id = 0; id < N5; id++) x[id] += dx[id];
        const double W_old = W;
        double vsq = 0.;
#pragma unroll
        for (int id = 1; id < 4; id++)
#pragma unroll
            for (int jd = 1; jd < 4; jd++) vsq += g.gcov[id][jd] * x[U1 + id - 1] * x[U1 + jd - 1];
        const double gsqtmp = 1. + vsq;
        e = eos.at(x[RHO], x[UU]);
        if (eos.tabulated())
            W = gsqtmp * (x[UU] + x[RHO] + e.p);
        else
            W = gsqtmp * (eos.gam * x[UU] + x[RHO]);
        errx = (W == 0.) ? fabs(W - W_old) : fabs(fdiv(W - W_old, W));
        if ((fabs(errx) <= NEWT_TOL) && (f <= 1.e-4) && (doing_extra == 0)) doing_extra = 1;
        if (doing_extra == 1) i_extra++;
        if (((fabs(errx) <= NEWT_TOL) && (doing_extra == 0)) || (i_extra > EXTRA_NEWT_ITER) ||
            (n_iter >= (MAX_NEWT_ITER - 1)))
            keep = false;
        n_iter++;
    }
    n_iter_out = n_iter;
    eos.refresh(g);
    int ret = 0;
    if (!isfinite(f) || !isfinite(df))
        ret = 2;
    else if ((fabs(errx) > MIN_NEWT_TOL) || (f > 1.e-4))
        ret = 1;
    if (ret) return 100 * ret + 1;
    if ((x[RHO] < 0.0) || (x[UU] < 0.0)) return 5;
    double pt[NPR];
#pragma unroll
    for (int k = 0; k < N5; k++) pt[k] = x[k];
#pragma unroll
    for (int k = B1; k <= B3; k++) pt[k] = prim[k];
    double gamma_tmp;
    if (gamma_calc_g5(pt, g, gamma_tmp) == 1) return 4;
#pragma unroll
    for (int k = 0; k < N5; k++) prim[k] = x[k];
    return 0;
}

}  // namespace harm

namespace harm {

// The tabulated EOS as a policy of the physics templates (harm_phys.hpp):
// mhd_calc_CoolEOS's pressure (phys.c:122-141) and the tabulated branch of
// vchar (phys.c:359-378): cs2 = (dp/drho + p/rho^2 dp/de) / h with e = u/rho,
// dp/de = rho dp/du, h = 1 + e + p/rho.  ref_derivs reproduces the reference's
// derivatives, whose finite-difference step (u hh / U_UNIT, cooleos.c:667-741)
// vanishes next to u in FP64 so that both are exactly 0.
struct EosTable {
    static constexpr bool TAB = true;
    EosTab t;
    int ref_derivs;
    __device__ EosPt at(double rho, double u) const
    {
        EosPt e;
        eos_table_p(t, rho, u, e.p, e.dpdrho, e.dpdu);
        return e;
    }
    __device__ double cs2(double rho, double u, const EosPt &pt) const
    {
        const double p = pt.p;
        double dpdrho = pt.dpdrho, dpdu = pt.dpdu;
        if (ref_derivs) {
            dpdrho = 0.;
            dpdu = 0.;
        }
        const double e = u / rho;
        const double enthalpy = 1.0 + e + p / rho;
        const double dpde = dpdu * rho;
        return (dpdrho + p / rho / rho * dpde) / enthalpy;
    }
};

}  // namespace harm
