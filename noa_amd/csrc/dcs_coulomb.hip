// Coulomb scattering of the PMS path on MI355X (src/noa/pms/dcs.hh:499-950):
//   coulomb_data       per K: centre-of-mass factors fCM [n][2], spin factor,
//                      screening parameters [n][9], inverse Wentzel path
//   coulomb_transport  per K: first two transport coefficients at a cutoff mu
//   hard_scattering    per K over a mixture of nel elements: cutoff angle mu0
//                      (Ridders' root, numerics.hh:154-214) and mean free
//                      path lb_h of elastic hard scatters
//   soft_scattering    per K: transverse transport of soft ionisation
//                      (closed form) plus photonuclear (a 102-node quadrature6
//                      of photonuclear * ratio * nu)
//
// The per-K functions are short and branchy, so they run one thread per K
// with the FP64 log/exp tables in LDS. Per-element values the reference
// recomputes in every call (pow(A, 1/3), pow(Z, 2/3), cos of the soft
// angle, the node values nu_j = 0.05 exp(t_j), which are the same for every
// K) are evaluated once on the host with the host libm. Soft scattering is
// one kernel too: a workgroup compacts the open photonuclear nodes of its K
// values in LDS, evaluates them in whole waves and sums them there. Every
// device function keeps the reference's operation order with FMA contraction
// off.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "capi_util.hh"
#include "dcs_consts.hh"
#include "dcs_tile.hh"
#include "fastmath.hh"

namespace noa_hip {

constexpr double KIN_CUTOFF = 1E-9;    // physics.hh:78
constexpr double EHS_PATH_MAX = 1E+9;  // physics.hh:79
constexpr double EHS_OVER_MSC = 1E-4;  // physics.hh:80
constexpr int NSF = 9;                 // physics.hh:87

constexpr int SOFT_ITV = 17;               // ceil(100 / 6) subintervals (dcs.hh:936, numerics.hh:80)
constexpr int SOFT_NODES = 6 * SOFT_ITV;   // 102
constexpr int SOFT_CHUNK = 16384;          // K values the workspace is sized for

// Nodes per workgroup (66 and 2 K values of the 23 nodes that can be open),
// and the number of K values up to which the open integrals are spread over
// lanes by node. A workgroup takes one K as long as 1024 of them fill the
// chip. Measured on MI355X (us, spread / not): 176 K 9.4 / 20, 1236 12 / 19,
// 2000 17 / 19, 4000 26 / 23, 16,384 82 / 48, 65,536 312 / 111.
constexpr int SOFT_TILE = 1536, SOFT_SPLIT_TILE = 64;
constexpr int64_t SOFT_SPLIT_MAX = 2048;

// Host-evaluated per-element values (bit-identical to the reference's).
struct CoulombElement {
    double A, I, Zd, mass;
    int32_t Z;
    double Ma;       // A * 0.931494
    double M2;       // (mass + Ma)^2
    double two_Ma;   // 2 Ma
    double mmMa;     // mass (mass + Ma)
    double rM2;      // (mass / Ma)^2
    double R1sq;     // (1.02934 A^(1/3) + 0.435)^2
    double s0_c;     // 5.179587126e-12 Z^(2/3)
    double wp_c;     // A * 2.54910918e8
};

CoulombElement make_coulomb_element(double A, double I, int32_t Z, double mass) {
    CoulombElement c{};
    c.A = A;
    c.I = I;
    c.Z = Z;
    c.Zd = double(Z);
    c.mass = mass;
    c.Ma = A * 0.931494;
    c.M2 = mass + c.Ma;
    c.M2 *= c.M2;
    c.two_Ma = 2. * c.Ma;
    c.mmMa = mass * (mass + c.Ma);
    c.rM2 = mass / c.Ma;
    c.rM2 *= c.rM2;
    const double R1 = 1.02934 * std::pow(A, 1. / 3) + 0.435;
    c.R1sq = R1 * R1;
    c.s0_c = 5.179587126E-12 * std::pow(double(Z), 2. / 3.);
    c.wp_c = A * 2.54910918E+08;
    return c;
}

// ---- per-K closed forms (dcs.hh:499-602) ----

__device__ __forceinline__ void coulomb_data_one(double K, const CoulombElement& c, double* fCM, double* s,
                                                 double* fspin, double* invlambda, const fm::Tab& t) {
#pragma clang fp contract(off)
    const double mass = c.mass;
    // dcs.hh:499-521
    const double s_inv = 1. / sqrt(c.M2 + c.two_Ma * K);
    fCM[0] = (K + mass + c.Ma) * s_inv;
    double k0 = (K * c.Ma + c.mmMa) * s_inv - mass;
    if (k0 < KIN_CUTOFF) k0 = KIN_CUTOFF;
    const double etot = K + mass + c.Ma;
    const double beta2 = K * (K + 2. * mass) / (etot * etot);
    fCM[1] = sqrt(c.rM2 * (1. - beta2) + beta2);
    // dcs.hh:524-527 at k0
    const double e = k0 + mass;
    *fspin = k0 * (e + mass) / (e * e);
    // dcs.hh:540-602 at k0
    const double p2 = k0 * (k0 + 2. * mass);
    const double d = 5.8406E-02 / p2;
    s[1] = d / c.R1sq;
    s[2] = d / 4.;
    const double ZE = c.Zd * e;
    const double zeta2 = 5.3251346E-05 * (ZE * ZE) / p2;
    double cK;
    if (zeta2 > 1.) {
        const int32_t terms = 10 + c.Z;
        double f = 0.;
        for (int32_t i = 1; i <= terms; i++) f += zeta2 / (double(i) * (double(i * i) + zeta2));
        cK = fm::exp(f, t);
    } else {
        cK = fm::exp(1. - 1. / (1. + zeta2) + zeta2 * (0.2021 + zeta2 * (0.0083 * zeta2 - 0.0369)), t);
    }
    const double cM = 1. + 3.34 * zeta2;
    double r = k0 / e;
    r *= r;
    const double cc = r * cK + (1. - r) * cM;
    const double s0 = c.s0_c * cc / p2;
    s[0] = s0;
    const double d01 = 1. / (s0 - s[1]);
    const double d02 = 1. / (s0 - s[2]);
    const double d12 = 1. / (s[1] - s[2]);
    s[6] = d01 * d01 * d02 * d02;
    s[7] = d01 * d01 * d12 * d12;
    s[8] = d12 * d12 * d02 * d02;
    s[3] = 2. * s[6] * (d01 + d02);
    s[4] = 2. * s[7] * (d12 - d01);
    s[5] = -2. * s[8] * (d12 + d02);
    // dcs.hh:530-537 (Wentzel path at s0)
    const double dw = k0 * (k0 + 2. * mass) / (c.Zd * (k0 + mass));
    *invlambda = 1. / (c.wp_c * s0 * (1. + s0) * dw * dw);
}

// dcs.hh:624-674.
__device__ __forceinline__ void transport_one(const double* s, double fspin, double mu, double* G,
                                              const fm::Tab& t) {
#pragma clang fp contract(off)
    const double nuc = (s[1] < s[2]) ? s[1] : s[2];
    if (mu < 1E-08 * nuc) {
        const double L = fm::log(1. + mu / s[0], t);
        const double r = mu / (mu + s[0]);
        const double k = s[0] * (1. + s[0]);
        G[0] = k * (r / s[0] - fspin * (L - r));
        const double I2 = mu - s[0] * (r - 2. * L);
        G[1] = 2. * k * (L - r - fspin * I2);
        return;
    }
    const double half_mu2 = 0.5 * mu * mu;
    double g0 = 0., g1 = 0.;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double si = s[i];
        double r = mu / (mu + si);
        double L = fm::log(1. + mu / si, t);
        double mu1 = mu;
        const double I0 = r / si;
        const double J0 = L;
        const double I1 = L - r;
        r *= si;
        L *= si;
        const double J1 = mu1 - L;
        const double I2 = mu1 - 2. * L + r;
        L *= si;
        mu1 *= si;
        const double J2 = half_mu2 + L - mu1;
        g0 += s[3 + i] * (J0 - fspin * J1) + s[6 + i] * (I0 - fspin * I1);
        g1 += s[3 + i] * (J1 - fspin * J2) + s[6 + i] * (I1 - fspin * I2);
    }
    const double k = s[0] * (1. + s[0]) * s[1] * s[1] * s[2] * s[2];
    G[0] = g0 * k;
    G[1] = g1 * (2. * k);
}

// Screening parameters for which the quotients and logarithms of
// restricted_cs have positive normal operands and results at any 0 <= mu < 1
// (NaN fails): there a division is fm::div_rn by the correctly rounded
// reciprocal and the logarithm fm::log_pos, the same values without the IEEE
// sequence (whose VCC use serialises the poles) and without special arguments.
__device__ __forceinline__ bool screening_ordinary(const double* s) {
    return s[0] >= 1e-100 && s[0] <= 1e100 && s[1] >= 1e-100 && s[1] <= 1e100 && s[2] >= 1e-100 && s[2] <= 1e100;
}

template <bool Fast>
__device__ __forceinline__ double cs_div(double a, double b) {
    if constexpr (Fast) return fm::div_rn(a, b, fm::recip_pos(b));
    else return a / b;
}
template <bool Fast>
__device__ __forceinline__ double cs_log(double x, const fm::Tab& t) {
    if constexpr (Fast) return fm::log_pos(x, t);
    else return fm::log(x, t);
}

// dcs.hh:697-735.
template <bool Fast>
__device__ __forceinline__ double restricted_cs(double mu, double fspin, const double* s, const fm::Tab& t) {
#pragma clang fp contract(off)
    if (mu >= 1.) return 0.;
    const double nuc = (s[1] < s[2]) ? s[1] : s[2];
    if (mu < 1E-08 * nuc) {
        const double L = cs_log<Fast>(cs_div<Fast>(s[0] + 1., s[0] + mu), t);
        const double r = cs_div<Fast>(1. - mu, (s[0] + mu) * (s[0] + 1.));
        const double k = s[0] * (1. + s[0]);
        return k * (r - fspin * (L - s[0] * r));
    }
    double cs = 0.;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double si = s[i];
        const double L = cs_log<Fast>(cs_div<Fast>(si + 1., si + mu), t);
        const double r = cs_div<Fast>(1. - mu, (si + mu) * (si + 1.));
        const double I1 = L - si * r;
        const double J1 = mu - si * L;
        cs += s[3 + i] * (L - fspin * J1) + s[6 + i] * (r - fspin * I1);
    }
    const double k = s[0] * (1. + s[0]) * s[1] * s[1] * s[2] * s[2];
    return k * cs;
}

struct Mixture {
    const double* G;
    const double* fCM;
    const double* screen;
    const double* invlambda;
    const double* fspin;
    int64_t nel, nkin;
};

// One kinetic energy of a mixture, shared by a group of L lanes (a power of
// two): lane l of the group holds the values of elements l, L + l, ..., (E - 1)
// L + l and evaluates those elements' terms; every sum over the elements is
// then taken in element order from the group's lanes, so that all of them hold
// the serial loop's value. Elements from L E on are read as they are needed.
template <int L, int E>
struct MixtureK {
    const Mixture& m;
    int64_t i;
    int lane;            // this lane's place in the group
    double s[E][NSF];    // its elements' screening parameters
    double fspin[E], invlambda[E];
    bool ordinary;       // screening_ordinary for all of them

    __device__ __forceinline__ MixtureK(const Mixture& mix, int64_t idx, int l) : m(mix), i(idx), lane(l) {
#pragma unroll
        for (int k = 0; k < E; k++) load(k * L + l, s[k], &fspin[k], &invlambda[k]);
        ordinary = true;
#pragma unroll
        for (int k = 0; k < E; k++) ordinary = ordinary && screening_ordinary(s[k]);
    }

    // (an element beyond the mixture reads the first one's values, unused)
    __device__ __forceinline__ void load(int64_t e, double* sc, double* sp, double* il) const {
        const int64_t o = (e < m.nel ? e : 0) * m.nkin + i;
#pragma unroll
        for (int k = 0; k < NSF; k++) sc[k] = m.screen[NSF * o + k];
        *sp = m.fspin[o];
        *il = m.invlambda[o];
    }

    // acc + the terms of elements first, first + 1, ... of the group's lanes
    __device__ __forceinline__ double add_in_order(double acc, double term, int64_t first) const {
#pragma clang fp contract(off)
        if constexpr (L == 1) return first < m.nel ? acc + term : acc;
#pragma unroll
        for (int l = 0; l < L; l++) {
            const double t = __shfl(term, l, L);
            if (first + l < m.nel) acc += t;
        }
        return acc;
    }

    // dcs.hh:737-751
    __device__ __forceinline__ double objective(double cs_h, double mu, const fm::Tab& t) const {
#pragma clang fp contract(off)
        double term[E];
        if (ordinary && mu >= 0.) {
#pragma unroll
            for (int k = 0; k < E; k++) term[k] = invlambda[k] * restricted_cs<true>(mu, fspin[k], s[k], t);
        } else {
#pragma unroll
            for (int k = 0; k < E; k++) term[k] = invlambda[k] * restricted_cs<false>(mu, fspin[k], s[k], t);
        }
        double cs = 0.;
#pragma unroll
        for (int k = 0; k < E; k++) cs = add_in_order(cs, term[k], k * L);
        for (int64_t e0 = L * E; e0 < m.nel; e0 += L) {
            double sc[NSF], sp, il;
            load(e0 + lane, sc, &sp, &il);
            cs = add_in_order(cs, il * restricted_cs<false>(mu, sp, sc, t), e0);
        }
        return cs - cs_h;
    }
};

// numerics.hh:154-214, with the end values given; false where the
// reference returns std::nullopt.
template <class M>
__device__ __forceinline__ bool ridders(double xa, double xb, double fa, double fb, double xtol, double rtol,
                                        uint32_t max_iter, double cs_h, const M& m, const fm::Tab& t, double* root) {
#pragma clang fp contract(off)
    if (fa * fb > 0) return false;
    if (fa == 0) { *root = xa; return true; }
    if (fb == 0) { *root = xb; return true; }
    const double tol = xtol + rtol * fmin(fabs(xa), fabs(xb));
    for (uint32_t it = 0; it < max_iter; it++) {
        double dm = 0.5 * (xb - xa);
        const double xm = xa + dm;
        const double fm_ = m.objective(cs_h, xm, t);
        double sgn = (fb > fa) ? 1. : -1.;
        double dn = sgn * dm * fm_ / sqrt(fm_ * fm_ - fa * fb);
        sgn = (dn > 0.) ? 1. : -1.;
        dn = fabs(dn);
        dm = fabs(dm) - 0.5 * tol;
        if (dn < dm) dm = dn;
        const double xn = xm - sgn * dm;
        const double fn = m.objective(cs_h, xn, t);
        if (fn * fm_ < 0.0) {
            xa = xn; fa = fn; xb = xm; fb = fm_;
        } else if (fn * fa < 0.0) {
            xb = xn; fb = fn;
        } else {
            xa = xn; fa = fn;
        }
        if (fn == 0.0 || fabs(xb - xa) < tol) { *root = xn; return true; }
    }
    return false;
}

// dcs.hh:753-838. All lanes of the group get the result.
template <int L, int E>
__device__ __forceinline__ void hard_one(const Mixture& mix, int64_t i, int lane, double max_mu0, double* mu0_out,
                                         double* lb_h_out, const fm::Tab& t) {
#pragma clang fp contract(off)
    const MixtureK<L, E> m(mix, i, lane);
    double invlb_m = 0., invlb1_m = 0., s_m_l = 0., s_m_h = 0.;
    for (int64_t e0 = 0; e0 < mix.nel; e0 += L) {
        const int64_t o = (e0 + lane < mix.nel ? e0 + lane : 0) * mix.nkin + i;
        const double invlb = mix.invlambda[o];
        const double scr = mix.screen[NSF * o];
        const double d = 1. / (mix.fCM[2 * o] * (1. + mix.fCM[1 + 2 * o]));
        invlb_m = m.add_in_order(invlb_m, invlb * mix.G[2 * o], e0);
        s_m_h = m.add_in_order(s_m_h, scr * invlb, e0);
        s_m_l = m.add_in_order(s_m_l, invlb / scr, e0);
        invlb1_m = m.add_in_order(invlb1_m, invlb * mix.G[1 + 2 * o] * d * d, e0);
    }
    const double lb_m = 1. / invlb_m;
    double lb_h = fmin(EHS_OVER_MSC / invlb1_m, EHS_PATH_MAX);
    double mu0;
    if (lb_m < lb_h) {
        const double s_m = (lb_h > 2. * lb_m) ? s_m_h * lb_m : 1. / (s_m_l * lb_m);
        mu0 = s_m * (lb_h - lb_m) / (s_m * lb_h + lb_m);
        const double cs_h = 1. / lb_h;
        double mu_max = fmin(4. * mu0, 1.);
        double mu_min = 0.25 * mu0;
        double fmax = m.objective(cs_h, mu_max, t), fmin_;
        if (fmax > 0.) {
            // as in the reference, mu0 and lb_h keep their estimates here
        } else {
            fmin_ = m.objective(cs_h, mu_min, t);
            if (fmin_ < 0.) {
                mu_max = mu_min;
                fmax = fmin_;
                mu_min = 0.;
                fmin_ = m.objective(cs_h, mu_min, t);
            }
            if (mu_min < max_mu0) {
                mu_max = fmin(mu_max, max_mu0);
                double root;
                if (ridders(mu_min, mu_max, fmin_, fmax, 1E-6 * mu0, 1E-6, 100, cs_h, m, t, &root)) mu0 = root;
            }
            mu0 = fmin(mu0, max_mu0);
            lb_h = m.objective(cs_h, mu0, t) + cs_h;
            lb_h = (lb_h <= 1. / EHS_PATH_MAX) ? EHS_PATH_MAX : 1. / lb_h;
        }
    } else {
        lb_h = lb_m;
        mu0 = 0;
    }
    *mu0_out = mu0;
    *lb_h_out = lb_h;
}

// dcs.hh:874-897.
__device__ __forceinline__ double transverse_ionisation(double K, const CoulombElement& c, const fm::Tab& t) {
#pragma clang fp contract(off)
    const double mass = c.mass, me = ELECTRON_MASS;
    const double p2 = K * (K + 2. * mass);
    const double E = K + mass;
    const double Wmax = 2. * me * p2 / (mass * mass + me * (me + 2. * E));
    const double W0 = 2. * p2 / me;
    const double mu_max = Wmax / W0;
    double mu3 = K * X_FRACTION / W0;
    if (mu3 > mu_max) mu3 = mu_max;
    const double mu2 = 0.62 * c.I / W0;
    if (mu2 >= mu3) return 0.;
    const double a0 = 0.5 * W0 / p2;
    const double a1 = -1. / Wmax;
    const double a2 = E * E / (W0 * p2);
    const double cs0 = 1.535336E-05 / c.A;
    return 2. * cs0 * c.Zd * (0.5 * a0 * (mu3 * mu3 - mu2 * mu2) + a1 * (mu3 - mu2) + a2 * fm::log(mu3 / mu2, t));
}

// dcs.hh:910-932: the mu-integrated ratio at one node.
__device__ __forceinline__ double photo_ratio(double K, double q, double mass, const fm::Tab& t) {
#pragma clang fp contract(off)
    const double E = K + mass;
    const double m02 = 0.4;
    const double q2 = q * q;
    const double tmax = 1.876544 * q;
    const double tmin = q2 * mass * mass / (E * (E - q));
    const double b1 = 1. / (1. - q2 / m02);
    const double c1 = 1. / (1. - m02 / q2);
    double L1 = b1 * fm::log((q2 + tmax) / (q2 + tmin), t);
    double L2 = c1 * fm::log((m02 + tmax) / (m02 + tmin), t);
    const double I0 = fm::log(tmax / tmin, t) - L1 - L2;
    L1 *= q2;
    L2 *= m02;
    const double I1 = L1 + L2;
    L1 *= q2;
    L2 *= m02;
    const double I2 = (tmax - tmin) * (b1 * q2 + c1 * m02) - L1 - L2;
    return (I1 * tmax - I2) / ((I0 * tmax - I1) * K * (K + 2. * mass));
}

// ---- kernels ----

// The log/exp tables in LDS as `tab`, visible after the next barrier.
#define NOA_FM_TABLES()                                                                          \
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES]; \
    load_fm_tables(fm_block);                                                                    \
    const fm::Tab tab = fm::tab_from_block(fm_block)
#define NOA_FM_PROLOGUE() \
    NOA_FM_TABLES();      \
    __syncthreads()

#define NOA_GRID_LOOP(i, n) \
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < (n); i += int64_t(gridDim.x) * blockDim.x)

__global__ __launch_bounds__(256) void coulomb_data_kernel(const double* __restrict__ K, int64_t n, CoulombElement c,
                                                           double* __restrict__ fCM, double* __restrict__ screen,
                                                           double* __restrict__ fspin,
                                                           double* __restrict__ invlambda) {
    NOA_FM_PROLOGUE();
    NOA_GRID_LOOP(i, n) {
        double f[2], s[NSF], sp, il;
        coulomb_data_one(K[i], c, f, s, &sp, &il, tab);
        fCM[2 * i] = f[0];
        fCM[2 * i + 1] = f[1];
#pragma unroll
        for (int k = 0; k < NSF; k++) screen[NSF * i + k] = s[k];
        fspin[i] = sp;
        invlambda[i] = il;
    }
}

__global__ __launch_bounds__(256) void coulomb_transport_kernel(const double* __restrict__ screen,
                                                                const double* __restrict__ fspin,
                                                                const double* __restrict__ mu, int64_t n_mu,
                                                                int64_t n, double* __restrict__ G) {
    NOA_FM_PROLOGUE();
    NOA_GRID_LOOP(i, n) {
        double s[NSF], g[2];
#pragma unroll
        for (int k = 0; k < NSF; k++) s[k] = screen[NSF * i + k];
        transport_one(s, fspin[i], mu[n_mu == 1 ? 0 : i], g, tab);
        G[2 * i] = g[0];
        G[2 * i + 1] = g[1];
    }
}

// What bounds it is the length of a K's chain of ~17 evaluations of the
// objective, one after the other, each three poles per element. One thread per
// K that read its elements' 11 values from memory in each evaluation took 96
// us for 65,536 K of three elements (74 with the first element's values in
// registers); held in registers, with the divisions and logarithms that
// restricted_cs needs no special cases for, 44 us.
template <int L, int E>
__global__ __launch_bounds__(256) void hard_scattering_kernel(Mixture m, double max_mu0, double* __restrict__ mu0,
                                                              double* __restrict__ lb_h) {
    NOA_FM_PROLOGUE();
    const int lane = threadIdx.x % L;
    // (the lanes of a group share i, so they leave the loop together)
    NOA_GRID_LOOP(v, m.nkin * L) {
        const int64_t i = v / L;
        double a, b;
        hard_one<L, E>(m, i, lane, max_mu0, &a, &b, tab);
        if (lane == 0) {
            mu0[i] = a;
            lb_h[i] = b;
        }
    }
}

struct SoftNodes {
    double nu[SOFT_NODES];  // X_FRACTION exp(t_j), host libm
    double h;               // subinterval width in t
    int32_t first;          // the nodes before this one have nu below the photonuclear model's 2e-3
    double q_pole;          // sqrt(m0^2), the q whose square is m0^2: photo_ratio is 0 / 0 there
    float pole_at, per_ln;  // K's subinterval that holds it: pole_at - per_ln ln K
};

// numerics.hh:91-108 weights.
static __constant__ double SOFT_W[6] = {0.08566225, 0.18038079, 0.23395697, 0.23395697, 0.18038079, 0.08566225};

// Node j's term of the integral, given its photonuclear DCS.
__device__ __forceinline__ double soft_term(double k, double nu, double dcs, int j, double h, double mass,
                                            const fm::Tab& t) {
#pragma clang fp contract(off)
    return dcs * photo_ratio(k, nu * k, mass, t) * nu * h * SOFT_W[j % 6];
}

// A workgroup's nodes in LDS, by item: node first + j of K slot k at k nb + j.
template <int TILE, bool SPLIT>
struct SoftLds {
    double nu[SOFT_NODES];
    double K[TILE];
    double term[TILE];
    uint16_t list[TILE];
    uint8_t whole[TILE];  // K slots whose nodes are all summed
    uint32_t n_open;
    // (SPLIT) the open integrals' shared values and node terms, by list entry
    double x9[9];
    F64::PhotoPre pre[SPLIT ? TILE : 1];
    double f[SPLIT ? 9 * TILE : 1];
};

__device__ double soft_all_nodes(double k, const SoftNodes& sn, double mass, const DcsConsts& c, const fm::Tab& t) {
#pragma clang fp contract(off)
    double acc = 0.;
#pragma unroll 1
    for (int j = 0; j < SOFT_NODES; j++) {
        const double q = sn.nu[j] * k;
        acc += soft_term(k, sn.nu[j], F64::photo_active(k, q, c) ? F64::photo(k, q, c, t) : 0., j, sn.h, mass, t);
    }
    return acc;
}

// One workgroup per `group` K values.
//
// The photonuclear DCS is zero below nu = 2e-3 (and q = 1 GeV), so of an
// ordinary K's 102 nodes only the last SOFT_NODES - first (23) can count and
// the others' transport ratios need not be formed; those of K above ~500 GeV
// all do. K outside [1e-20, 1e30] GeV and NaN, and masses outside it, where a
// ratio might overflow and carry its NaN into the sum, take all nodes in the
// reference's order (soft_all_nodes), and so does a K one of whose nodes falls
// on the pole of the ratio.
//
// Bound: FP64 VALU issue, ~4500 instructions per open node. Open nodes are
// compacted in LDS and drained by whole waves; SPLIT spreads each over 9
// lanes by quadrature node, for calls with too few K values to fill the chip.
// Measured for 65,536 K: 111 us, against 733 us when the 102 nodes of each K
// went through memory as (K, q) pairs of a map and one thread per K formed
// their 102 ratios (64 workgroups per pass of 16,384 K); 9.4 us for 176 K.
template <int TILE, bool SPLIT>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(SPLIT ? 3 : 4))) void soft_kernel(
    const double* __restrict__ K, int64_t n, DcsConsts, CoulombElement ce, SoftNodes sn, int32_t group,
    double* __restrict__ out) {
    __shared__ SoftLds<TILE, SPLIT> s;
    NOA_FM_TABLES();
    const ConstsPtr cp = vector_kernarg_consts();
    const int tid = threadIdx.x;
    const int64_t k0 = int64_t(blockIdx.x) * group;
    const int nk = int(n - k0 < group ? n - k0 : group);
    const int first = sn.first, nb = SOFT_NODES - first;
    for (int j = tid; j < SOFT_NODES; j += WG) s.nu[j] = sn.nu[j];
    for (int kk = tid; kk < nk; kk += WG) s.K[kk] = K[k0 + kk];
    if (SPLIT && tid < 9) s.x9[tid] = GL9_X[tid];
    if (tid == 0) s.n_open = 0;
    __syncthreads();
    for (int kk = tid; kk < nk; kk += WG) {
        const double k = s.K[kk];
        // (in range also where K is NaN)
        const int itv = int(fminf(fmaxf(sn.pole_at - sn.per_ln * __logf(float(k)), 0.f), float(SOFT_ITV - 1)));
        bool whole = !(k >= 1e-20 && k <= 1e30 && ce.mass >= 1e-20 && ce.mass <= 1e30);
#pragma unroll
        for (int m = 0; m < 6; m++) whole |= s.nu[6 * itv + m] * k == sn.q_pole;
        s.whole[kk] = whole;
    }
#pragma unroll 1
    for (int i0 = 0; i0 < nk * nb; i0 += WG) {
        const DcsConsts& c = item_consts(cp);
        const int i = i0 + tid;
        bool open = false;
        if (i < nk * nb) {
            const int kk = i / nb;
            const double k = s.K[kk];
            open = F64::photo_active(k, s.nu[first + (i - kk * nb)] * k, c);
            s.term[i] = 0.;
        }
        wave_append(open, &s.n_open, s.list, uint32_t(i));
    }
    __syncthreads();
    const uint32_t n_open = s.n_open;
    if constexpr (SPLIT) {
        for (uint32_t e = tid; e < n_open; e += WG) {
            const DcsConsts& c = item_consts(cp);
            const uint32_t i = s.list[e], kk = i / uint32_t(nb), j = first + (i - kk * nb);
            const double k = s.K[kk];
            s.pre[e] = F64::photo_setup<false, true>(k, s.nu[j] * k, c, tab);
        }
        __syncthreads();
        for (uint32_t v = tid; v < 9 * n_open; v += WG) {
            const DcsConsts& c = item_consts(cp);
            const uint32_t e = v / 9;
            const F64::PhotoPre p = s.pre[e];
            s.f[v] = F64::photo_node<false, true>(p, s.x9[v - 9 * e], c, tab);
        }
        __syncthreads();
    }
#pragma unroll 1
    for (uint32_t e = tid; e < n_open; e += WG) {
        const DcsConsts& c = item_consts(cp);
        const uint32_t i = s.list[e], kk = i / uint32_t(nb), j = first + (i - kk * nb);
        const double k = s.K[kk], nu = s.nu[j];
        double d;
        if (!SPLIT || !(c.fast_ok && k + c.mass <= F64::FAST_E_MAX)) {
            d = F64::photo(k, nu * k, c, tab);
        } else {
            d = 0.;
            for (int m = 0; m < 9; m++) d = F64::photo_add<false>(s.f[9 * e + m], GL9_W[m], d);
            d = F64::photo_finish<false, true>(k, s.pre[e], d, c);
        }
        s.term[i] = soft_term(k, nu, d, int(j), sn.h, ce.mass, tab);
    }
    __syncthreads();
    // 8 lanes per K: strided sums, then a fixed-order tree
    for (int v = tid; v < nk * 8; v += WG) {
        const int kk = v >> 3;
        double acc = 0.;
        for (int j = v & 7; j < nb; j += 8) acc += s.term[kk * nb + j];
        acc += __shfl_xor(acc, 4, 8);
        acc += __shfl_xor(acc, 2, 8);
        acc += __shfl_xor(acc, 1, 8);
        if ((v & 7) == 0) {
            const DcsConsts& c = item_consts(cp);
            const double k = s.K[kk];
            if (s.whole[kk]) acc = soft_all_nodes(k, sn, ce.mass, c, tab);
            out[k0 + kk] = transverse_ionisation(k, ce, tab) + 2. * acc;
        }
    }
}

// Lanes per K and elements per lane of the hard-scattering kernel for nel
// elements at n energies. Few energies: one element per lane (up to 8 lanes),
// the shortest chain. Once its waves exceed two per SIMD, as few lanes as hold
// the mixture in registers (3 elements each), since every lane of a group
// repeats the root search around its elements' terms. Measured (us, spread /
// held): 3 elements 64 K 22 / 43, 65,536 K 54 / 44, 262,144 K 188 / 132; 5
// elements 64 K 22 / 42, 65,536 K 90 / 63; 1 element 65,536 K 20.5.
struct HardShape {
    int lanes, elements;
};
inline HardShape hard_shape(int64_t nel, int64_t n) {
    const int spread = nel <= 1 ? 1 : nel <= 2 ? 2 : nel <= 4 ? 4 : 8;
    if (n * spread <= 131072 || nel > 12) return {spread, 1};
    if (nel <= 3) return {1, int(nel)};
    if (nel <= 6) return {2, nel == 4 ? 2 : 3};
    return {4, nel <= 8 ? 2 : 3};
}

// K values per workgroup of the soft-scattering kernel, of which a tile holds
// `room`: equal shares for the fewest whole rounds of the 1024 workgroups that
// the chip holds. About half of the nodes are open and a workgroup drains them
// 256 at a time, so a small group leaves most lanes of its last pass idle.
// Measured (us; 22 K values per workgroup / up to 66 / up to 66 in equal
// shares): 65,536 K 119 / 110 / 110, 70,000 125 / 131 / 120, 100,000 168 / 171 /
// 163, 2^20 1509 / 1279 / 1273.
int32_t soft_group(int64_t n, int64_t room) {
    const int64_t round = 1024 * std::max<int64_t>(1, room);
    const int64_t slots = 1024 * ((n + round - 1) / round);
    return int32_t((n + slots - 1) / slots);
}

unsigned grid_for(int64_t n) { return unsigned(std::max<int64_t>(1, std::min<int64_t>(65536, (n + 255) / 256))); }

}  // namespace noa_hip

using namespace noa_hip;

extern "C" {

int noa_dcs_coulomb_data_f64(const double* K, int64_t n, const noa_dcs_element* element, double mass, double* fCM,
                             double* screening, double* fspin, double* invlambda, hipStream_t stream) {
    if (int rc = check_element(element, mass)) return rc;
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (n == 0) return ok();
    if (!K || !fCM || !screening || !fspin || !invlambda)
        return fail(NOA_DCS_EINVAL, "K, fCM, screening, fspin and invlambda must all be non-NULL");
    const CoulombElement c = make_coulomb_element(element->A, element->I, element->Z, mass);
    hipLaunchKernelGGL(coulomb_data_kernel, dim3(grid_for(n)), dim3(256), 0, stream, K, n, c, fCM, screening, fspin,
                       invlambda);
    if (int rc = check_hip(hipGetLastError(), "coulomb_data_kernel")) return rc;
    return ok();
}

int noa_dcs_coulomb_transport_f64(const double* screening, const double* fspin, const double* mu, int64_t n_mu,
                                  int64_t n, double* G, hipStream_t stream) {
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (!(n_mu == 1 || n_mu == n)) return fail(NOA_DCS_EINVAL, "mu must hold 1 or n values (got %lld, n = %lld)",
                                               (long long)n_mu, (long long)n);
    if (n == 0) return ok();
    if (!screening || !fspin || !mu || !G) return fail(NOA_DCS_EINVAL, "screening, fspin, mu and G must be non-NULL");
    hipLaunchKernelGGL(coulomb_transport_kernel, dim3(grid_for(n)), dim3(256), 0, stream, screening, fspin, mu, n_mu,
                       n, G);
    if (int rc = check_hip(hipGetLastError(), "coulomb_transport_kernel")) return rc;
    return ok();
}

int noa_dcs_hard_scattering_f64(int64_t nel, int64_t nkin, const double* G, const double* fCM,
                                const double* screening, const double* invlambda, const double* fspin, double* mu0,
                                double* lb_h, hipStream_t stream) {
    if (nel < 1) return fail(NOA_DCS_EINVAL, "nel must be >= 1");
    if (nkin < 0) return fail(NOA_DCS_EINVAL, "nkin must be >= 0");
    if (nkin == 0) return ok();
    if (!G || !fCM || !screening || !invlambda || !fspin || !mu0 || !lb_h)
        return fail(NOA_DCS_EINVAL, "every array argument must be non-NULL");
    // physics.hh:81-84, with the host libm as in the reference
    const double max_mu0 = 0.5 * (1. - std::cos(1E+00 * M_PI / 180.));
    const Mixture m{G, fCM, screening, invlambda, fspin, nel, nkin};
    const HardShape shape = hard_shape(nel, nkin);
    const int lanes = shape.lanes;
    auto* kernel = &hard_scattering_kernel<1, 1>;
    if (lanes == 1) {
        if (shape.elements == 2) kernel = &hard_scattering_kernel<1, 2>;
        if (shape.elements == 3) kernel = &hard_scattering_kernel<1, 3>;
    } else if (lanes == 2) {
        kernel = shape.elements == 1   ? &hard_scattering_kernel<2, 1>
                 : shape.elements == 2 ? &hard_scattering_kernel<2, 2>
                                       : &hard_scattering_kernel<2, 3>;
    } else if (lanes == 4) {
        kernel = shape.elements == 1   ? &hard_scattering_kernel<4, 1>
                 : shape.elements == 2 ? &hard_scattering_kernel<4, 2>
                                       : &hard_scattering_kernel<4, 3>;
    } else {
        kernel = &hard_scattering_kernel<8, 1>;
    }
    hipLaunchKernelGGL(kernel, dim3(grid_for(nkin * lanes)), dim3(256), 0, stream, m, max_mu0, mu0, lb_h);
    if (int rc = check_hip(hipGetLastError(), "hard_scattering_kernel")) return rc;
    return ok();
}

}  // extern "C"

namespace {

int check_soft_args(const double* K, int64_t n, const noa_dcs_element* element, double mass, const double* result) {
    if (int rc = check_element(element, mass)) return rc;
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (n > 0 && (!K || !result)) return fail(NOA_DCS_EINVAL, "K and result must be non-NULL");
    return NOA_DCS_OK;
}

int soft_run(const double* K, int64_t n, const noa_dcs_element* element, double mass, double* result,
             hipStream_t stream) {
    // numerics.hh:72-108 on [ln 1e-6, 0] with min_points = 100 (dcs.hh:905-936)
    SoftNodes sn{};
    const double lb = std::log(1E-06);
    sn.h = (0. - lb) / double(uint32_t(SOFT_ITV));
    const double x6[6] = {0.03376524, 0.16939531, 0.38069041, 0.61930959, 0.83060469, 0.96623476};
    for (int j = 0; j < SOFT_NODES; j++)
        sn.nu[j] = X_FRACTION * std::exp(lb + sn.h * (double(uint32_t(j / 6)) + x6[j % 6]));
    sn.q_pole = std::sqrt(0.4);
    sn.per_ln = float(1. / sn.h);
    sn.pole_at = float((std::log(sn.q_pole / X_FRACTION) - lb) / sn.h);
    sn.first = 0;
    while (sn.first < SOFT_NODES && sn.nu[sn.first] < 2E-03 * (1. - 1E-09)) sn.first++;
    const CoulombElement ce = make_coulomb_element(element->A, element->I, element->Z, mass);
    const DcsConsts c = make_consts(element->A, element->I, element->Z, mass);
    const int nb = SOFT_NODES - sn.first;
    constexpr int64_t most = int64_t(1) << 30;
    for (int64_t k0 = 0; k0 < n; k0 += most) {
        const int64_t nK = std::min<int64_t>(most, n - k0);
        const bool split = nK <= SOFT_SPLIT_MAX;
        const int32_t group = soft_group(nK, (split ? SOFT_SPLIT_TILE : SOFT_TILE) / nb);
        const auto kernel = split ? &soft_kernel<SOFT_SPLIT_TILE, true> : &soft_kernel<SOFT_TILE, false>;
        hipLaunchKernelGGL(kernel, dim3(unsigned((nK + group - 1) / group)), dim3(WG), 0, stream, K + k0, nK, c, ce, sn,
                           group, result + k0);
        if (int rc = check_hip(hipGetLastError(), "soft_kernel")) return rc;
    }
    return ok();
}

}  // namespace

extern "C" {

int64_t noa_dcs_soft_scattering_workspace_bytes(int64_t n) {
    if (n <= 0) return 0;
    return std::min<int64_t>(n, SOFT_CHUNK) * SOFT_NODES * int64_t(3 * sizeof(double));
}

int noa_dcs_soft_scattering_f64(const double* K, int64_t n, const noa_dcs_element* element, double mass,
                                double* result, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
    if (int rc = check_soft_args(K, n, element, mass, result)) return rc;
    if (n == 0) return ok();
    if (!workspace || workspace_bytes < noa_dcs_soft_scattering_workspace_bytes(n))
        return fail(NOA_DCS_EINVAL, "workspace must hold noa_dcs_soft_scattering_workspace_bytes(n) bytes");
    return soft_run(K, n, element, mass, result, stream);
}

int noa_dcs_soft_scattering_f64_noalloc(const double* K, int64_t n, const noa_dcs_element* element, double mass,
                                        double* result, hipStream_t stream) {
    if (int rc = check_soft_args(K, n, element, mass, result)) return rc;
    if (n == 0) return ok();
    return soft_run(K, n, element, mass, result, stream);
}

}  // extern "C"
