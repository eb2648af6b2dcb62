// harm_nse.hpp -- one point of the cooling-table generator: lepton and
// nucleon densities, the chemical (n <-> p) equilibrium, neutrino cooling
// rates and optical depths, and the total EOS, over harm_fermi.hpp.
//
// The chain is written once over a policy that says who forms the quadrature
// nodes: NseSerial (one thread, host or device) or NseWave (a block of three
// wavefronts per point).  Both add the same terms in the same order.
//
// Follows number_den.f90 (fxnn, fxnp, lepton, neta, peta, eeta),
// mnewtf.f90 (mnewt with ludcmp/lubksb, here for the one-unknown systems the
// chain solves), neu_rate.f90 (pair, urca, brem, plasmon), accretion.f90
// (opt_dep), chem_eq.f90 (chem_eq, eqnucl, nuclear, funcnb, neutrino,
// rtbis_funcnb) and abundance.f90 (the table point).  Integer powers x**n
// are evaluated as the oracle build of the reference (amdflang -O2) compiles
// them: left-to-right products up to the 8th power, binary powering above
// (gfortran's powi uses binary powering throughout, so a gfortran build can
// differ in the last bit).  Undecorated literals keep their single-precision
// values (0.23, 13.8, 0.557, 0.3, 1./3.).
#pragma once
#include "harm_fermi.hpp"

namespace harm {

// 40-point Gauss-Legendre positive nodes and weights (gauss_legendre,
// gauss_integral.f90:118-219), and the 20-point Laguerre rule of FermiRules
// (gauss_laguerre, gauss_integral.f90:26-113).
struct NseRules {
    FermiRules f;
    double lx40[20], lw40[20];
};

// The nodes as the sums below walk them, {abscissa, weight} each: fd the 80 of
// a Fermi-Dirac integral (three 20-point Legendre intervals on (-1, 1), then
// the Laguerre tail), rate the 80 of the beta rates (40-point Legendre for
// n -> p, 20-point Laguerre for p + e- and for n + e+).
struct NseNodes {
    double fd[80][2], rate[80][2];
};

inline void nse_nodes(const NseRules &R, NseNodes &N)
{
    for (int q = 0; q < 3; q++)
        for (int j = 0; j < 10; j++)
            for (int s = 0; s < 2; s++) {
                N.fd[20 * q + 2 * j + s][0] = s ? -R.f.lx[j] : R.f.lx[j];
                N.fd[20 * q + 2 * j + s][1] = R.f.lw[j];
            }
    for (int j = 0; j < 20; j++) {
        for (int s = 0; s < 2; s++) {
            N.rate[2 * j + s][0] = s ? -R.lx40[j] : R.lx40[j];
            N.rate[2 * j + s][1] = R.lw40[j];
        }
        N.fd[60 + j][0] = N.rate[40 + j][0] = N.rate[60 + j][0] = R.f.gx[j];
        N.fd[60 + j][1] = N.rate[40 + j][1] = N.rate[60 + j][1] = R.f.gw[j];
    }
}

HD double ipow(double x, int n)
{
    if (n <= 8) {
        double r = x;
        for (int i = 1; i < n; i++) r = r * x;
        return r;
    }
    double res = 1.0, sq = x;
    bool have = false;
    while (n) {
        if (n & 1) {
            res = have ? res * sq : sq;
            have = true;
        }
        n >>= 1;
        if (n) sq = sq * sq;
    }
    return res;
}

constexpr double NSE_SQRT2 = 1.4142135623730951;  // dsqrt(2.0d0)

// Share v (0..7) of F_{1/2}, F_{3/2}, ..., F_{NK-1/2} at (eta, theta): ten of
// the 80 nodes of dfermi's quadrature (gauss_integral.f90:241-349), all of one
// subinterval.  The NK integrals have their nodes, occupation and square roots
// in common: x^k sqrt(1 + x theta / 2) is sqrt(x (1 + x theta / 2)) x^(k-1/2),
// and the first subinterval's z^2 = x only changes the weight, so a node costs
// one exp, one square root and one division whatever NK is.  The derivatives
// that dfermi also forms have no reader in the table point.
template <int NK>
HD void fd_share(const double (*nd)[2], int v, double eta, double theta, double (&acc)[NK])
{
    double s1, s2, s3;
    fd_breaks(eta, s1, s2, s3);
    const int seg = v >> 1;
    double c, h;
    if (seg == 0) {
        h = 0.5 * sqrt(s1);
        c = h;
    } else if (seg == 1) {
        c = 0.5 * (s1 + s2);
        h = 0.5 * (s2 - s1);
    } else if (seg == 2) {
        c = 0.5 * (s2 + s3);
        h = 0.5 * (s3 - s2);
    } else {
        c = s3;
        h = 1.0;
    }
    for (int k = 0; k < NK; k++) acc[k] = 0.0;
#pragma unroll 2
    for (int i = 0; i < 10; i++) {
        const double *n = nd[10 * v + i];
        const double z = c + h * n[0];
        const double x = (seg == 0) ? z * z : z;
        const double w = (seg == 0) ? 2.0 * z * n[1] : n[1];
        // 1 / (exp(x - eta) + 1) without overflow on either side
        const double d = x - eta, t = exp(-fabs(d));
        double f = w * sqrt(x * (1.0 + 0.5 * x * theta)) * ((d > 0.0) ? t : 1.0) / (1.0 + t);
#pragma unroll
        for (int k = 0; k < NK; k++) {
            acc[k] = acc[k] + f;
            f = f * x;
        }
    }
#pragma unroll
    for (int k = 0; k < NK; k++) acc[k] = acc[k] * h;
}

// What one node of the beta rates contributes (the URCA integrands
// neu_rate.f90 func1-3 and chem_eq.f90 func1k..func3r share abscissae and
// factors): gk, gr = weight x sqrt(x^2 - 1/beta^2) base^2 times the occupation
// of the forward and of the reverse reaction, base = q - x, x - q or x + q,
// y = 1 / (exp(.) + 1) of the neutrino blocking.
struct RateNode {
    double gk, gr, base, y;
    int kind;  // 0 n -> p, 1 p + e-, 2 n + e+; -1 none
};

HD RateNode nse_rate_node(const double *n, int id, double xkt, double xetae, double xetaep)
{
    RateNode r;
    r.kind = id < 40 ? 0 : (id < 60 ? 1 : 2);
    const double betae = xkt / FD_XME, q = (FD_XMN - FD_XMP) / xkt, ib = 1.0 / betae;
    double x, xe, arg;
    if (r.kind == 0) {
        const double a = FD_XME / xkt;
        x = 0.5 * (a + q) + 0.5 * (q - a) * n[0];
        xe = xetae - (x - ib);
        arg = r.base = q - x;
    } else if (r.kind == 1) {
        x = q + n[0];
        xe = -xetae + (x - ib);
        arg = r.base = x - q;
    } else {
        x = FD_XME / xkt + n[0];
        xe = -xetaep + (x - ib);
        arg = r.base = x + q;
    }
    r.y = 1.0 / (exp(arg) + 1.0);
    const double t = exp(-fabs(xe)), o = 1.0 / (1.0 + t);
    const double g = n[1] * x * sqrt(x * x - 1.0 / (betae * betae)) * r.base * r.base;
    r.gk = g * ((xe > 0.0) ? t * o : o);
    r.gr = g * ((xe > 0.0) ? o : t * o);
    return r;
}

// One thread forms every node (host, or one table point per device thread).
struct NseSerial {
    const NseNodes &N;
    static constexpr int NR = 80;
    HD explicit NseSerial(const NseNodes &n) : N(n) {}
    HD bool writes() const { return true; }

    // F[s][k] for the sets s in the mask
    template <int NS, int NK>
    HD void moments(const double (&eta)[NS], const double (&theta)[NS], unsigned mask, double (&F)[NS][NK]) const
    {
        for (int s = 0; s < NS; s++) {
            if (!(mask >> s & 1u)) continue;
            double a[8][NK];
            for (int v = 0; v < 8; v++) fd_share<NK>(N.fd, v, eta[s], theta[s], a[v]);
            for (int k = 0; k < NK; k++)
                F[s][k] = ((a[0][k] + a[1][k]) + (a[2][k] + a[3][k])) + ((a[4][k] + a[5][k]) + (a[6][k] + a[7][k]));
        }
    }
    HD void rate_nodes(double xkt, double xetae, double xetaep, RateNode (&r)[NR]) const
    {
        for (int i = 0; i < NR; i++) r[i] = nse_rate_node(N.rate[i], i, xkt, xetae, xetaep);
    }
    // s[kind] = sum of f(node) over that kind's nodes
    template <class F>
    HD void rate_sums(const RateNode (&r)[NR], F f, double (&s)[3]) const
    {
        for (int q = 0; q < 3; q++) {
            double v[64];
            for (int i = 0; i < 64; i++) v[i] = 0.0;
            for (int i = 0; i < NR; i++)
                if (r[i].kind == q) v[i < 60 ? i : i - 60] = f(r[i]);
            for (int o = 32; o > 0; o >>= 1)
                for (int i = 0; i < o; i++) v[i] = v[i] + v[i + o];
            s[q] = v[0];
        }
    }
    template <class F>
    HD void three(double x0, double x1, double x2, F f, double &f0, double &f1, double &f2) const
    {
        f0 = f(x0);
        f1 = f(x1);
        f2 = f(x2);
    }
};

#if defined(__HIPCC__)
// A block of three wavefronts per point.  A wavefront is 8 groups of 8 lanes,
// one (eta, theta) per group and ten nodes per lane, so the six densities of a
// Newton step on two species (value and the two of its central difference
// each) are one pass; the three wavefronts take the three abscissae of the
// outer Newton's central difference.  Every lane holds the point's scalars.
struct NseWave {
    const double (*fd)[2];    // node tables and exchange in LDS
    const double (*rate)[2];
    double *ex;               // [3]
    static constexpr int NR = 2;
    __device__ bool writes() const { return threadIdx.x < 64; }

    static __device__ double dpp(double v, const int ctrl_sel)
    {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        int lo = (int)b, hi = (int)(b >> 32);
        if (ctrl_sel == 0) {
            lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, false);  // lane ^ 1
            hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, false);
        } else if (ctrl_sel == 1) {
            lo = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xF, 0xF, false);  // lane ^ 2
            hi = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xF, 0xF, false);
        } else {
            lo = __builtin_amdgcn_mov_dpp(lo, 0x141, 0xF, 0xF, false);  // the other half of 8 lanes
            hi = __builtin_amdgcn_mov_dpp(hi, 0x141, 0xF, 0xF, false);
        }
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
    }
    static __device__ double lane_value(double v, int lane)
    {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
    template <int NS, int NK>
    __device__ void moments(const double (&eta)[NS], const double (&theta)[NS], unsigned, double (&F)[NS][NK]) const
    {
        static_assert(NS <= 8, "a wavefront holds 8 sets");
        const int lane = (int)(threadIdx.x & 63u), g = lane >> 3;
        double e = eta[0], t = theta[0];
#pragma unroll
        for (int s = 1; s < NS; s++)
            if (g == s) {
                e = eta[s];
                t = theta[s];
            }
        double a[NK];
        fd_share<NK>(fd, lane & 7, e, t, a);
#pragma unroll
        for (int k = 0; k < NK; k++) {
            a[k] = a[k] + dpp(a[k], 0);
            a[k] = a[k] + dpp(a[k], 1);
            a[k] = a[k] + dpp(a[k], 2);
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int k = 0; k < NK; k++) F[s][k] = lane_value(a[k], 8 * s);
    }
    __device__ void rate_nodes(double xkt, double xetae, double xetaep, RateNode (&r)[NR]) const
    {
        const int lane = (int)(threadIdx.x & 63u);
        r[0].kind = r[1].kind = -1;
        if (lane < 60) r[0] = nse_rate_node(rate[lane], lane, xkt, xetae, xetaep);
        if (lane < 20) r[1] = nse_rate_node(rate[60 + lane], 60 + lane, xkt, xetae, xetaep);
    }
    template <class F>
    __device__ void rate_sums(const RateNode (&r)[NR], F f, double (&s)[3]) const
    {
        s[0] = (r[0].kind == 0) ? f(r[0]) : 0.0;
        s[1] = (r[0].kind == 1) ? f(r[0]) : 0.0;
        s[2] = (r[1].kind == 2) ? f(r[1]) : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int q = 0; q < 3; q++) s[q] = s[q] + __shfl_xor(s[q], o, 64);
    }
    template <class F>
    __device__ void three(double x0, double x1, double x2, F f, double &f0, double &f1, double &f2) const
    {
        const int w = (int)(threadIdx.x >> 6);
        const double v = f(w == 0 ? x0 : (w == 1 ? x1 : x2));
        __syncthreads();  // the values of the trial before have been read
        if ((threadIdx.x & 63u) == 0) ex[w] = v;
        __syncthreads();
        f0 = ex[0];
        f1 = ex[1];
        f2 = ex[2];
    }
};
#endif

// mnewt (mnewtf.f90:97-151) for one unknown, one trial at a time: ludcmp of
// the 1x1 Jacobian is singular when it is zero (or NaN), and then the step is
// fvec itself.  Where the tolerances lie below the round-off of the function
// (the outer solve's 1e-8 of a density, against a relative rate imbalance) the
// trials settle into a cycle of a few values that runs on to ntrial: a trial
// depends on x alone, so once x comes back to an earlier value whole periods
// are stepped over, and the last trials give the x that all of them would
// (Brent's cycle search: the value to meet is renewed at trials 1, 2, 4, ...).
struct NseNewton {
    double x, xs;
    int k, ks, next;
    bool done;
    HD explicit NseNewton(double x0) : x(x0), xs(x0), k(0), ks(0), next(1), done(false) {}
    HD void trial(double fjac, double fvec, double tolx, double tolf, int ntrial)
    {
        if (fabs(fvec) <= tolf) {
            done = true;
            return;
        }
        if (fabs(fjac) > 0.) fvec = fvec / fjac;
        x = x + fvec;
        k++;
        if (fabs(fvec) <= tolx) {
            done = true;
            return;
        }
        if (x == xs) {
            const int p = k - ks;
            k += (ntrial - k) / p * p;
        } else if (k == next) {
            xs = x;
            ks = k;
            next *= 2;
        }
        if (k >= ntrial) done = true;
    }
};

// Step of the central differences of usrfun_neta / usrfun_peta / usrfun_eeta
// (number_den.f90): |x| 1e-8, at least 1e-50.
HD double nse_step(double x)
{
    const double xacc = fabs(x) * 1.0e-8;
    return xacc < 1.0e-50 ? 1.0e-50 : xacc;
}

// fvec and fjac of target - n from its values at x, x + xacc, x - xacc
HD void nse_difference(double target, double n0, double np_, double nm, double xacc, double &fjac, double &fvec)
{
    const double f = target - n0, fp = target - np_, fm = target - nm;
    fjac = (fp - fm) / (2.0 * xacc);
    fvec = -f;
}

// number_den.f90: the density of a Fermi species [fm^-3] is
// c (F_{1/2} + beta F_{3/2}) at (eta, beta = kT / m), with this c
HD double fd_density_c(double mass, double xkt)
{
    const double beta = xkt / mass, h = mass / FD_HC;
    return NSE_SQRT2 / (FD_PI * FD_PI) * ipow(h, 3) * pow(beta, 1.5);
}

HD double nse_tol(double n)
{
    const double tol = 1.0e-8 * n;
    return tol < 1.0e-50 ? 1.0e-50 : tol;
}

// nuclear (chem_eq.f90; peta, neta of number_den.f90): proton and neutron
// degeneracies for a proton fraction, the two Newton solves side by side
template <class P>
HD void nuclear(const P &pol, double xkt, double xnb, double xp, double &xetan, double &xetap)
{
    double tp = xnb * xp, tn = xnb - tp;
    if (tp <= 0.0) tp = 0.0;
    if (tn <= 0.0) tn = 0.0;
    const double bp = xkt / FD_XMP, bn = xkt / FD_XMN;
    const double cp = fd_density_c(FD_XMP, xkt), cn = fd_density_c(FD_XMN, xkt);
    NseNewton a(-10.0), b(-10.0);
    while (!(a.done && b.done)) {
        const double da = nse_step(a.x), db = nse_step(b.x);
        const double eta[6] = {a.x, a.x + da, a.x - da, b.x, b.x + db, b.x - db};
        const double th[6] = {bp, bp, bp, bn, bn, bn};
        double F[6][2], fj, fv;
        pol.template moments<6, 2>(eta, th, (a.done ? 0u : 7u) | (b.done ? 0u : 56u), F);
        if (!a.done) {
            nse_difference(tp, cp * (F[0][0] + bp * F[0][1]), cp * (F[1][0] + bp * F[1][1]),
                           cp * (F[2][0] + bp * F[2][1]), da, fj, fv);
            a.trial(fj, fv, 1.0e-20, nse_tol(tp), 200);
        }
        if (!b.done) {
            nse_difference(tn, cn * (F[3][0] + bn * F[3][1]), cn * (F[4][0] + bn * F[4][1]),
                           cn * (F[5][0] + bn * F[5][1]), db, fj, fv);
            b.trial(fj, fv, 1.0e-20, nse_tol(tn), 200);
        }
    }
    xetap = a.x;
    xetan = b.x;
}

// eeta (number_den.f90:303-323): electron degeneracy for a net lepton density
// (lepton, number_den.f90:372-395)
template <class P>
HD double eeta(const P &pol, double xkt, double xne)
{
    const double be = xkt / FD_XME, c = fd_density_c(FD_XME, xkt), tol = nse_tol(xne);
    NseNewton s(0.510998910 / xkt);
    while (!s.done) {
        const double d = nse_step(s.x), xe[3] = {s.x, s.x + d, s.x - d};
        double eta[6], th[6], F[6][2], nl[3], fj, fv;
#pragma unroll
        for (int q = 0; q < 3; q++) {
            eta[q] = xe[q];
            eta[3 + q] = -xe[q] - (double)2.0f / be;
            th[q] = th[3 + q] = be;
        }
        pol.template moments<6, 2>(eta, th, 63u, F);
#pragma unroll
        for (int q = 0; q < 3; q++) nl[q] = c * (F[q][0] + be * F[q][1]) - c * (F[3 + q][0] + be * F[3 + q][1]);
        nse_difference(xne, nl[0], nl[1], nl[2], d, fj, fv);
        s.trial(fj, fv, 1.0e-20, tol, 200);
    }
    return s.x > 0.0 ? 0.0 : s.x;
}

// pair (neu_rate.f90:18-96): e+e- annihilation emissivities of one electron
// and one other flavour, from F_{1/2} .. F_{7/2} of electrons and positrons
HD void pair_rates(double betae, const double *Fe, const double *Fp, double &ev1, double &ev2)
{
    constexpr double QC = 1.023e23;
    double cv = 2.0 * 0.23 + 0.5, ca = 0.5;
    const double cv1e = cv * cv + ca * ca, cv2e = cv * cv - ca * ca;
    cv = 2.0 * 0.23 - 0.5;
    ca = -0.5;
    const double cv1m = cv * cv + ca * ca, cv2m = cv * cv - ca * ca;
    auto moments = [&](const double *F, double &m_1, double &m0, double &m1, double &m2) {
        m_1 = F[0];
        m0 = F[0] + betae * F[1];
        m1 = F[0] + 2.0 * betae * F[1] + betae * betae * F[2];
        m2 = F[0] + 3.0 * betae * F[1] + 3.0 * betae * betae * F[2] + ipow(betae, 3) * F[3];
    };
    double u_1, u0, u1, u2, fai_1, fai0, fai1, fai2;
    moments(Fe, u_1, u0, u1, u2);
    moments(Fp, fai_1, fai0, fai1, fai2);
    const double pre = QC / (36.0 * FD_PI) * (2.0 / ipow(FD_PI, 4)) * ipow(betae, 3);
    const double A = 8.0 * (fai1 * u2 + fai2 * u1) - 2.0 * (fai_1 * u2 + fai2 * u_1) + 7.0 * (fai0 * u1 + fai1 * u0) +
                     5.0 * (fai0 * u_1 + fai_1 * u0);
    const double B = fai0 * (u1 + u_1) + (fai_1 + fai1) * u0;
    ev1 = pre * (cv1e * A + 9.0 * cv2e * B);
    ev2 = pre * (cv1m * A + 9.0 * cv2m * B);
}

// brem, plasmon (neu_rate.f90:208-259)
HD double brem(double nb, double xkt)
{
    const double rho10 = nb * 1.66e5, t11 = xkt * 1.16059e-1;
    return 3.35e27 * pow(rho10, 2.0) * pow(t11, 5.5);
}

HD double plasmon(double xkt, double xetae)
{
    const double t11 = xkt * 1.16059e-1, etae = xetae + 0.510998910 / xkt;
    const double gp = 5.565e-2 * sqrt((FD_PI * FD_PI + 3.0 * (etae * etae)) / 3.0);
    return 1.5e32 * ipow(t11, 9) * ipow(gp, 6) * exp(-gp) * (1.0 + gp) * (2.0 + (gp * gp) / (1.0 + gp));
}

// A point's densities for the chemical equilibrium (common /nucl/, chem_eq.f90).
struct NuclCommon {
    double xnnucl, xkt, xne0, HdFac, nb0;
};

// The gas at a proton fraction: what abundance() writes out, and the relative
// imbalance of the n <-> p rates that chem_eq brings to zero.
struct NseState {
    double e1, p1, b1, b2, ta1, ta2, ts, xnee, xnep, imbalance;
};

// funcnb (chem_eq.f90) and the second half of abundance (abundance.f90:130-
// 200), which form the same things: degeneracies, densities, EOS (eos.f90),
// the ten passes of the neutrino trapping (eos_neu, h_dep, opt_dep, b_neu,
// accretion.f90) and neutrino (chem_eq.f90).  The electrons', positrons',
// protons' and neutrons' integrals are one pass, and the emissivities, which
// no trapping pass changes, are formed once.
template <class P>
HD_CALL void nse_state(const P &pol, const NuclCommon &c, double xp, double nhe, NseState &o)
{
    const double xkt = c.xkt, betae = xkt / FD_XME, t11 = xkt * 1.16059e-1;
    const double betap = xkt / FD_XMP, betan = xkt / FD_XMN;
    double xetan, xetap;
    nuclear(pol, xkt, c.xnnucl, xp, xetan, xetap);
    const double xnp = c.xnnucl * xp, xnn = c.xnnucl - xnp, xne = c.xnnucl * xp + c.xne0;
    const double xetae = eeta(pol, xkt, xne);
    const double xetaep = -xetae - (double)2.0f / betae;
    double F[4][4];
    {
        const double eta[4] = {xetae, xetaep, xetap, xetan}, th[4] = {betae, betae, betap, betan};
        pol.template moments<4, 4>(eta, th, 15u, F);
    }
    const double cden = fd_density_c(FD_XME, xkt);
    o.xnee = cden * (F[0][0] + betae * F[0][1]);
    o.xnep = cden * (F[1][0] + betae * F[1][1]);
    // eos_npe (eos.f90:31-113), eos_rad, eos_he
    constexpr double c23 = (double)(2.0f / 3.0f), c32 = (double)(3.0f / 2.0f);
    const double pi2 = FD_PI * FD_PI;
    const double he = FD_XME / FD_HC, hp = FD_XMP / FD_HC, hn = FD_XMN / FD_HC;
    const double cpe = c23 * sqrt(2.0) / pi2 * (he * he * he) * FD_XME * pow(betae, 2.5);
    const double cpp = c23 * sqrt(2.0) / pi2 * (hp * hp * hp) * FD_XMP * pow(betap, 2.5);
    const double cpn = c23 * sqrt(2.0) / pi2 * (hn * hn * hn) * FD_XMN * pow(betan, 2.5);
    auto pres = [](double cp, double b, const double *f) { return cp * (f[1] + 0.5 * b * f[2]); };
    auto ener = [](double ce, double b, const double *f) { return ce * (f[1] + b * f[2]); };
    const bool pos = o.xnee > 0.0;
    const double p = pres(cpe, betae, F[0]) + (pos ? pres(cpe, betae, F[1]) : 0.0) + pres(cpp, betap, F[2]) +
                     pres(cpn, betan, F[3]);
    const double e = ener(c32 * cpe, betae, F[0]) + (pos ? ener(c32 * cpe, betae, F[1]) : 0.0) +
                     ener(c32 * cpp, betap, F[2]) + ener(c32 * cpn, betan, F[3]);
    double er, pr, sr, ehe, phe, she;
    eos_rad(xkt, er, pr, sr);
    eos_he(xkt, nhe, ehe, phe, she);
    o.p1 = p + pr + phe;
    o.e1 = e + er + ehe;
    // opt_dep's emissivities (accretion.f90:63-98): pair, urca, brem, plasmon
    double ev1, ev2, s[3];
    pair_rates(betae, F[0], F[1], ev1, ev2);
    RateNode nodes[P::NR];
    pol.rate_nodes(xkt, xetae, xetaep, nodes);
    pol.rate_sums(nodes, [](const RateNode &r) { return r.gk * r.base; }, s);
    const double hlf = 0.5 * ((FD_XMN - FD_XMP) / xkt - FD_XME / xkt), t6 = ipow(t11, 6);
    const double evn_k = 1.14473926e37 * t6 * xnn * (s[0] * hlf);
    const double evep_k = 1.14473926e37 * t6 * xnp * s[1];
    const double even_k = 1.14473926e37 * t6 * xnn * s[2];
    const double evbrem = brem(c.xnnucl, xkt), evplasmon = plasmon(xkt, xetae);
    const double qe = ev1 + evep_k + even_k + evn_k + evbrem / 3.0 + evplasmon;
    const double qo = ev2 + evbrem / 3.0;
    const double xl = 5.67051e39 * 4.0 * 7.0 / 8.0 * ipow(t11, 4);
    const double cv = (double)(0.5f + 2.0f * 0.23f), alph = 1.25;
    const double csn = (1.0 + 5.0 * (alph * alph)) / 24.0;
    const double csp = (4.0 * ((cv - 1.0) * (cv - 1.0)) + 5.0 * (alph * alph)) / 24.0;
    const double r = xkt / 0.510998910;
    double b1 = 0.0, b2 = 0.0;
    for (int i = 0; i < 10; i++) {
        double eneu, pneu, sneu;
        eos_neu(xkt, b1, b2, eneu, pneu, sneu);
        const double hd = h_dep(c.HdFac, c.nb0, o.p1 + pneu, o.e1 + eneu);
        o.ta1 = qe * hd / xl;
        o.ta2 = qo * hd / xl;
        o.ts = csn * 1.76e-5 * xnn * hd * (double)13.8f * (r * r) + csp * 1.76e-5 * xnp * hd * (double)13.8f * (r * r);
        const double b1o = b1, b2o = b2;
        b_neu(o.ta1, o.ta2, o.ts, b1, b2);
        if (b1 == b1o && b2 == b2o) break;  // the passes left would repeat this one
    }
    o.b1 = b1;
    o.b2 = b2;
    // neutrino (chem_eq.f90): forward and reverse rates of each reaction
    pol.rate_sums(nodes, [b1](const RateNode &q) { return q.gk * fabs(1.0 - b1 * q.y) + q.gr * fabs(b1 * q.y); }, s);
    const double t5 = ipow(t11, 5), mn = xnn < 0.0 ? 0.0 : xnn, mp = xnp < 0.0 ? 0.0 : xnp;
    const double rn = 2.03813046e35 * t5 * mn * (s[0] * hlf), rep = 2.03813046e35 * t5 * mp * s[1];
    const double ren = 2.03813046e35 * t5 * mn * s[2];
    o.imbalance = (fabs(rep) < 1.0e-80) ? (rep - ren - rn) / (fabs(rep) + 1.0e-80) : (rep - ren - rn) / fabs(rep);
}

// abundance (abundance.f90:6-243) with chem_eq and eqnucl (chem_eq.f90; the
// equilibrium proton fraction by Newton, rtbis_funcnb): one table point.
// rho [g cm^-3], T [K]; out: e, p [erg cm^-3], Qnu [erg cm^-2 s^-1], tau, and
// the pair densities [fm^-3].
template <class P>
HD void abundance(const P &pol, double rho, double T, double HdFac, double (&out)[6])
{
    const double xnb = rho / 1.66e15, xkt = T / 1.16059e10;
    const double xnuc0 = xnuc(xnb, xkt), nnuc = xnb * xnuc0, nhe = (xnb - nnuc) / 4.0;
    NuclCommon c;
    c.nb0 = xnb;
    c.xnnucl = nnuc;
    c.xne0 = fabs(1.0 - xnuc0) * xnb / 2.0;
    c.HdFac = HdFac;
    c.xkt = xkt;
    const double tol = nse_tol(c.xnnucl);
    NseState st;
    NseNewton s(0.5);
    while (!s.done) {
        const double d = nse_step(s.x);
        double f0, f1, f2, fj, fv;
        pol.three(
            s.x, s.x + d, s.x - d,
            [&](double y) {
                nse_state(pol, c, y, c.xne0 / (double)2.0f, st);
                return st.imbalance;
            },
            f0, f1, f2);
        nse_difference(0.0, f0, f1, f2, d, fj, fv);
        s.trial(fj, fv, 1.0e-20, tol, 200);
    }
    if (!pol.writes()) return;
    double xp = s.x;
    if (xp < 0.0) xp = 0.0;
    if (xp > 1.0) xp = 1.0;
    nse_state(pol, c, xp, nhe, st);
    double eneu, pneu, sneu;
    eos_neu(xkt, st.b1, st.b2, eneu, pneu, sneu);
    const double c557 = (double)0.557f, c3 = (double)0.3f;
    out[0] = (st.e1 + eneu) * 1.6021772e33;
    out[1] = (st.p1 + pneu) * 1.6021772e33;
    out[2] = 7.0 / 8.0 * FD_SIGMASB * ipow(T, 4) / (double)0.75f *
             (1. / (0.5 * st.ta1 + 0.5 * st.ts + c557 + c3 / st.ta1) +
              1. / (0.5 * st.ta2 + 0.5 * st.ts + c557 + c3 / st.ta2));
    out[3] = st.ts + st.ta1 + st.ta2;
    out[4] = st.xnee;
    out[5] = st.xnep;
}

}  // namespace harm
