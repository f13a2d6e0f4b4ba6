// PUMAS v1.2.1 DCS tabulation on the GPU: the x = ln(q / K) grid and the
// per-row table of compute_dcs_table (src/noa/3rdparty/_pumas/pumas.c:
// 11693-11787) with its row fill dcs_tabulate_row (:11422-11507), for the
// default models PUMAS tabulates (pumas.c:190-198): SSR bremsstrahlung
// (:13979-14068), SSR pair production (:14458-14671, 12-point rule over the
// asymmetry) and DRSS photonuclear with the ALLM97 structure function
// (:14690-15146, 9-point log-scale rule over Q^2), through their m^2/kg
// wrappers (:11067-11112).
//
// One wave per table row (process, element, kinetic energy): each lane
// evaluates the DCS at its grid nodes (the 12- and 9-point integrals run
// inside the lane), the row's logarithms and abscissae go to LDS, and the
// lanes then take the PCHIP slopes (Fritsch-Butland interior, three-point
// ends and the linear first bin of math_pchip_initialise, pumas.c:10039-10088)
// and the envelope exponent. A second launch gives the rows below the first
// positive exponent of each process and element that exponent
// (pumas.c:11745-11761), and a third the envelope maxima (pumas.c:11526-11679,
// a search over the interpolated table; see pumas_envelope_kernel).
//
// FP64 throughout, with the table-driven log and exp of fastmath.hh (powers as
// exp of a multiple of the log); the grid is computed on the host with the
// reference's operations.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "capi_util.hh"
#include "fastmath.hh"
#include "launch_slices.hh"
#include "pumas_search.hh"

namespace noa_hip {
namespace pumas {

constexpr int MAX_X = 192;  // grid nodes: cutoff >= ~2e-12
constexpr int N_REVERSE = 20;
constexpr double X_REVERSE = 0.6;
constexpr double DXMIN = 1E-03;
constexpr double MAX_FRACTION = 0.95;
constexpr int N_MIN = 10;
constexpr int PER_DECADE = 15;

constexpr double ALPHA_EM = 7.2973525693E-03;
constexpr double HBAR_C = 1.973269804E-16;
constexpr double ELECTRON_MASS = 0.510998910E-03;
constexpr double PROTON_MASS = 0.938272;
constexpr double NEUTRON_MASS = 0.939565;
constexpr double PION_MASS = 0.13957018;
constexpr double AVOGADRO_NUMBER = 6.02214076E+23;
constexpr double PI = 3.14159265358979323846;
constexpr double INV_LN10 = 0.43429448190325182765;
constexpr double NUCLEON_MASS = 0.5 * (PROTON_MASS + NEUTRON_MASS);
// MeV-unit constants of the SSR models (pumas.c:13891-13894, 14461-14463)
constexpr double SSR_SQRTE = 1.648721270700128;
constexpr double SSR_ME = 0.5109989461;
constexpr double SSR_RE = 2.8179403227E-13;
constexpr double SSR_MMU = 105.6583745;
constexpr double PAIR_SQRTE = 1.6487212707;  // pumas.c:14298, 14633

// Gauss-Legendre nodes and weights on [0, 1] (the 9- and 12-point rows of
// pumas.c:12527-12614).
static __constant__ double GQ9_X[9] = {0.0159198802461870, 0.0819844463366821, 0.1933142836497048,
                                       0.3378732882980955, 0.5000000000000000, 0.6621267117019045,
                                       0.8066857163502952, 0.9180155536633179, 0.9840801197538130};
static __constant__ double GQ9_W[9] = {0.0406371941807872, 0.0903240803474287, 0.1303053482014677,
                                       0.1561735385200015, 0.1651196775006299, 0.1561735385200015,
                                       0.1303053482014677, 0.0903240803474287, 0.0406371941807872};
static __constant__ double GQ12_X[12] = {0.0092196828766404, 0.0479413718147625, 0.1150486629028477,
                                         0.2063410228566913, 0.3160842505009099, 0.4373832957442655,
                                         0.5626167042557344, 0.6839157494990901, 0.7936589771433087,
                                         0.8849513370971523, 0.9520586281852375, 0.9907803171233596};
static __constant__ double GQ12_W[12] = {0.0235876681932559, 0.0534696629976592, 0.0800391642716731,
                                         0.1015837133615330, 0.1167462682691774, 0.1245735229067014,
                                         0.1245735229067014, 0.1167462682691774, 0.1015837133615330,
                                         0.0800391642716731, 0.0534696629976592, 0.0235876681932559};

// Chebyshev coefficients of the real dilogarithm (CERNLIB RDILOG, C332), the
// series of pumas.c:12673-12738.
static __constant__ double DILOG_C[20] = {
    0.42996693560813697,  0.40975987533077105,  -0.01858843665014592, 0.00145751084062268,
    -0.00014304184442340, 0.00001588415541880,  -0.00000190784959387, 0.00000024195180854,
    -0.00000003193341274, 0.00000000434545063,  -0.00000000060578480, 0.00000000008612098,
    -0.00000000001244332, 0.00000000000182256,  -0.00000000000027007, 0.00000000000004042,
    -0.00000000000000610, 0.00000000000000093,  -0.00000000000000014, 0.00000000000000002};

struct Grid {
    double x[MAX_X];
    int32_t n;
    double cutoff;
};

// Launch invariants computed on the host with the host libm, the
// reference's: the element's powers and logarithms, the mass-dependent
// bremsstrahlung terms and the literal exponentials, so that every exit
// (q >= q_max, ...) is decided on the reference's values.
struct Globals {
    double e1, e05, e_16, e13, e_13;  // exp(1), exp(1/2), exp(-1/6), exp(1/3), exp(-1/3)
    double lq0;                       // log(Q0^2 / Lambda^2) of ALLM97
};

struct ElementConsts {
    double Z, A;
    double z13;         // Z^(1/3)
    double Z13m;        // Z^(-1/3)
    double Z23;         // Z^(2/3)
    double dn;          // 1.54 A^0.27
    double lnA;         // ln A
    double shadow_low;  // exp(-0.1 ln A)
    double b_delta1;    // the bremsstrahlung nuclear-size terms (pumas.c:14009-14016)
    double b_delta2;
};

// What is left of the launch invariants is computed where it is used, from
// these, with the host's operations: the kernel arguments have 4096 bytes.

// m (1 - 0.75 sqrt(e) Z^(1/3)): the highest energy loss is K plus this, with
// bremsstrahlung's sqrt(e) or pair production's.
__device__ __forceinline__ double q_offset(double mass, double sqrte, const ElementConsts& c) {
#pragma clang fp contract(off)
    return mass * (1. - 0.75 * sqrte * c.z13);
}

// Radiation logarithms by Z (pumas.c:13773-13802); 0 = use 182.7.
static __constant__ double RAD_LOG[92] = {
    202.4, 151.9, 159.9, 172.3, 177.9, 178.3, 176.6, 173.4, 170.0, 165.8, 165.8, 167.1, 169.1, 170.8, 172.2,
    173.4, 174.3, 174.8, 175.1, 175.6, 176.2, 176.8, 0.0,   0.0,   0.0,   175.8, 0.0,   0.0,   173.1, 0.0,
    0.0,   173.0, 0.0,   0.0,   173.5, 0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   175.9, 0.0,   0.0,   0.0,
    0.0,   0.0,   0.0,   0.0,   177.4, 0.0,   0.0,   178.6, 0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,
    0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   177.6, 0.0,
    0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   178.0, 0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,   0.0,
    0.0,   179.8};

// (Z is the same for the whole workgroup: a scalar load)
__device__ __forceinline__ double rad_log(double Z) {
    const int i = __builtin_amdgcn_readfirstlane((Z >= 1. && Z < 93.) ? int(Z) : 0);
    const double v = i ? RAD_LOG[i - 1] : 0.;
    return v > 0. ? v : 182.7;
}

constexpr int MAX_KERNARG = 4096;
constexpr int MAX_EL = 30;  // elements per table launch (kernel-argument budget)

struct ElementBlock {
    ElementConsts e[MAX_EL];
};

// The grid for the envelope kernel, which reads the nodes as floats only: the
// m evenly spaced ones are recomputed, which leaves room for more elements.
constexpr int MAX_ENV_EL = 48;

struct EnvelopeGrid {
    float tail[N_REVERSE];
    int32_t m;
    double x0, dx;
};

struct EnvelopeBlock {
    ElementConsts e[MAX_ENV_EL];
};

// The log/exp tables in LDS as `tb` (every thread of the workgroup calls it).
#define NOA_PUMAS_TABLES()                                                                                    \
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];             \
    for (unsigned i = threadIdx.x; i < fm::TABLE_DOUBLES; i += blockDim.x) fm_block[i] = fm::table_entry(int(i)); \
    __syncthreads();                                                                                          \
    const fm::Tab tb = fm::tab_from_block(fm_block)

// Li2(x) by the RDILOG reductions onto [0, 1] and the Clenshaw sum.
__device__ double dilog(double x, const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double PI3 = PI * PI / 3.;
    const double PI6 = PI * PI / 6.;
    const double PI12 = PI * PI / 12.;
    if (x == 10) return PI6;
    if ((x == -1.) || (1. - x == 0.)) return -PI12;
    const double T = -x;
    double A, S, Y;
    if (T > -1. && T < 0.) {
        // the range of both of pair production's arguments: the reductions on
        // either side of -0.5 as one, since the lanes of a wave take both
        const bool big = T <= -0.5;
        const double T1 = 1. + T;
        Y = (big ? -T1 : -T) / (big ? T : T1);
        S = big ? 1. : -1.;
        const double l = fm::log_sel(-T, tb), l1 = fm::log_sel(T1, tb);
        A = big ? -PI6 + l * (-0.5 * l + l1) : 0.5 * (l1 * l1);
    } else if (T <= -2) {
        Y = -1. / (1. + T);
        S = 1.;
        const double l1 = fm::log_sel(-T, tb), l2 = fm::log_sel(1. + 1. / T, tb);
        A = -PI3 + 0.5 * (l1 * l1 - l2 * l2);
    } else if (T < -1.) {
        Y = -1. - T;
        S = -1.;
        A = fm::log_sel(-T, tb);
        A = -PI6 + A * (A + fm::log_sel(1. + 1. / T, tb));
    } else if (T <= 1.) {
        Y = T;
        S = 1.;
        A = 0.;
    } else {
        Y = 1. / T;
        S = -1.;
        const double l = fm::log_sel(T, tb);
        A = PI6 + 0.5 * (l * l);
    }
    const double H = Y + Y - 1;
    const double ALFA = H + H;
    double B0 = 0., B1 = 0., B2 = 0.;
#pragma unroll
    for (int i = 19; i >= 0; i--) {
        B0 = DILOG_C[i] + ALFA * B1 - B2;
        B2 = B1;
        B1 = B0;
    }
    return -(S * (B0 - H * B2) + A);
}

// SSR bremsstrahlung, atomic DCS in m^2 / GeV (pumas.c:13979-14068).
__device__ double brems_ssr(const ElementConsts& c, double rl, const Globals& G, double m, double K, double q,
                            const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double Z = c.Z;
    if ((Z <= 0) || (c.A <= 0) || (m <= 0) || (K <= 0) || (q <= 0)) return 0.;
    if (q >= K + q_offset(m, SSR_SQRTE, c)) return 0.;
    const double energy = (K + m) * 1E+03;
    const double v = q * 1E+03 / energy;
    m *= 1E+03;
    const double Z13 = 1. / c.z13;
    const double rl_inel = (Z == 1.) ? 446. : 1429.;
    const double delta = m * m * v / (2. * energy * (1. - v));
    const double rz = rl * Z13;
    double phi1 = fm::log_sel(rz * (m / SSR_ME) / (1. + rz * G.e05 * delta / SSR_ME), tb);
    double phi2 = fm::log_sel(rz * G.e_16 * (m / SSR_ME) / (1. + rz * G.e13 * delta / SSR_ME), tb);
    const double iz = 1. - 1. / Z;
    phi1 -= c.b_delta1 * iz;
    phi2 -= c.b_delta2 * iz;
    const double s1 = fm::log_sel(m / delta / (m * delta / (SSR_ME * SSR_ME) + SSR_SQRTE), tb);
    const double s2 = fm::log_sel(1. + SSR_ME / (delta * rl_inel * Z13 * Z13 * SSR_SQRTE), tb);
    const double s_atomic = (4. / 3. * (1. - v) + v * v) * (s1 - s2);
    double s_rad;
    if (v < .0 || v > 1.) {
        s_rad = 0.;
    } else if (v < 0.02) {
        s_rad = -0.00349 + 148.84 * v + -987.531 * v * v;
    } else if (v < 0.1) {
        s_rad = 0.1642 + 132.573 * v + -585.361 * v * v + 1407.77 * v * v * v;
    } else if (v < 0.9) {
        s_rad = -2.8922 + -19.0156 * v + 57.698 * v * v;
        const double t = fm::log_sel(1. - v, tb);
        s_rad += -63.418 * v * fm::log_sel(v, tb) + 14.1166 * t + 1.84206 * t * t;
    } else {
        s_rad = 2134.19 + 581.823 * v + -2708.85 * v * v;
        const double t = fm::log_sel(1. - v, tb);
        s_rad += 4767.05 * v * fm::log_sel(v, tb) + 1.52918 * t + 0.361933 * t * t;
    }
    const double result =
        ((2. - 2. * v + v * v) * phi1 - 2. / 3. * (1. - v) * phi2) + 1. / Z * s_atomic + 0.25 * ALPHA_EM * phi1 * s_rad;
    if (result <= 0.) return 0.;
    const double aux = 2 * (SSR_ME / m) * SSR_RE * Z;
    return aux * aux * (ALPHA_EM / q) * result * 1E-04;
}

// The parts of the SSR pair DDCS (pumas.c:14466-14500) that do not depend
// on the asymmetry rho, for one (element, K, q).
struct PairQ {
    double v, m, energy, ev, rl, Z13, d_n, beta, xi0, pref, me_dn2, me_m2;
};

// The atomic-electron factor zeta of pair production (pumas.c:14482-14492),
// which depends on the element and K only.
__device__ __forceinline__ double pair_zeta(const ElementConsts& c, double m_gev, double K, const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double Z = c.Z;
    const double energy = (K + m_gev) * 1E+03;
    const double m = m_gev * 1E+03;
    double g1, g2;
    if (Z == 1.) {
        g1 = 4.4E-05;
        g2 = 4.8E-05;
    } else {
        g1 = 1.95E-05;
        g2 = 5.3E-05;
    }
    const double zeta1 = (0.073 * fm::log_sel(energy / m / (1. + g1 * c.Z23 * energy / m), tb) - 0.26);
    const double zeta2 = (0.058 * fm::log_sel(energy / m / (1 + g2 / c.Z13m * energy / m), tb) - 0.14);
    return ((zeta1 > 0.) && (zeta2 > 0.)) ? zeta1 / zeta2 : 0.;
}

__device__ __forceinline__ PairQ pair_setup(const ElementConsts& c, double rl, double m_gev, double K, double q,
                                            double zeta) {
#pragma clang fp contract(off)
    const double Z = c.Z;
    PairQ s;
    s.energy = (K + m_gev) * 1E+03;
    s.v = q / (K + m_gev);
    s.m = m_gev * 1E+03;
    s.ev = s.energy * s.v;
    s.rl = rl;
    const double are = ALPHA_EM * SSR_RE;
    const double const_prefactor = 4. / (3. * PI) * Z * (are * are);
    s.Z13 = c.Z13m;
    s.d_n = c.dn;
    s.pref = const_prefactor * (Z + zeta) * (1. - s.v) / s.v;
    s.beta = s.v * s.v / (2. * (1. - s.v));
    const double mv = s.m * s.v / (2. * SSR_ME);
    s.xi0 = mv * mv;
    const double a = SSR_ME / s.m * s.d_n;
    s.me_dn2 = a * a;
    const double b = SSR_ME / s.m;
    s.me_m2 = b * b;
    return s;
}

// SSR pair DDCS at the reference's rho (pumas.c:14499-14609).
__device__ double pair_d2_ssr(const PairQ& s, const Globals& G, double rho, const fm::Tab& tb) {
#pragma clang fp contract(off)
    rho = 1 - rho;
    const double rho2 = rho * rho;
    const double beta = s.beta;
    const double omr = 1. - rho2;
    const double xi = s.xi0 * omr / (1. - s.v);
    const double xi1 = 1. + xi;
    const double w = s.ev * omr;
    const double c05 = 2. * SSR_ME * G.e05 * s.rl * s.Z13 * xi1 / w;
    const double c13 = 2. * SSR_ME * G.e13 * s.rl * s.Z13 * xi1 / w;

    // electron diagram
    const double lxi_i = fm::log_sel(1. + 1. / xi, tb);
    const double Pe = (2. + rho2) * (1. + beta) + xi * (3. + rho2);
    const double Be = Pe * lxi_i + (1. - rho2 - beta) / xi1 - (3. + rho2);
    const double Ce2 = (omr * (1. + beta) + xi * (3. - rho2)) * lxi_i + 2. * (1. - beta - rho2) / xi1 - (3. - rho2);
    const double Ce1 = Be - Ce2;
    const double De = Pe * dilog(1. / xi1, tb) - (2. + rho2) * xi * lxi_i - (xi + rho2 + beta) / xi1;
    const double sx = s.rl * s.Z13 * sqrt(xi1);
    const double sx6 = s.rl * s.Z13 * G.e_16 * sqrt(xi1);
    const double re = De / Be;
    // the forms for re > 0 and re <= 0 share their logarithms (and the muon
    // diagram's): nodes of one wave take both
    const bool pe = re > 0.;
    const double Xe = (fabs(re) < 100) ? fm::exp(-fabs(re), tb) : 0.;
    const double be = pe ? Xe : 1.;
    const double fe = pe ? s.me_dn2 : Xe * s.me_dn2;
    const double ree = pe ? re : 0.5 * re;
    const double Le1 = fm::log_sel(sx / (be + (pe ? c05 : Xe * c05)), tb) - ree - 0.5 * fm::log_sel(be + fe * xi1, tb);
    const double Le2 = fm::log_sel(sx6 / (be + (pe ? c13 : Xe * c13)), tb) - ree - 0.5 * fm::log_sel(be + fe * G.e_13 * xi1, tb);
    double diagram_e = s.pref * (Ce1 * Le1 + Ce2 * Le2);
    if (diagram_e < 0.) diagram_e = 0.;

    // muon diagram
    const double lxi = fm::log_sel(xi1, tb);
    const double b15 = 1. + (3. * beta) / 2.;
    const double Pm = (1. + rho2) * b15 - 1. / xi * (1. + 2. * beta) * omr;
    const double Bm = Pm * lxi + xi * (1. - rho2 - beta) / xi1 + (1. + 2. * beta) * omr;
    const double Cm2 = ((1. - beta) * omr - xi * (1. + rho2)) * lxi / xi - 2. * (1. - beta - rho2) / xi1 + 1. - beta -
                       (1. + beta) * rho2;
    const double Cm1 = Bm - Cm2;
    const double Dm = Pm * dilog(xi / xi1, tb) + b15 * omr / xi * lxi +
                      (1. - rho2 - beta / 2. * (1. + rho2) + omr / (2. * xi) * beta) * xi / xi1;
    const double num = s.m / SSR_ME * s.rl * s.Z13 / s.d_n;
    const double rm = Dm / Bm;
    const bool pm = rm > 0.;
    const double Xm = (fabs(rm) < 100) ? fm::exp(-fabs(rm), tb) : 0.;
    const double bm = pm ? Xm : 1.;
    const double rmm = pm ? rm : 0.;
    const double Lm1 = fm::log_sel(num / (bm + (pm ? c05 : c05 * Xm)), tb) - rmm;
    const double Lm2 = fm::log_sel(num / (bm + (pm ? c13 : c13 * Xm)), tb) - rmm;
    double diagram_mu = s.pref * s.me_m2 * (Cm1 * Lm1 + Cm2 * Lm2);
    if (diagram_mu < 0.) diagram_mu = 0.;
    return (diagram_e + diagram_mu) * 1E-01 / s.energy;
}

// SSR pair production, atomic DCS in m^2 / GeV (pumas.c:14624-14671): the
// 12-point rule over t = ln(rho) on [ln(1 - rmax), 0].
__device__ double pair_ssr(const ElementConsts& c, double rl, const Globals& G, double mass, double K, double q,
                           const fm::Tab& tb) {
#pragma clang fp contract(off)
    if ((c.Z <= 0) || (c.A <= 0) || (mass <= 0) || (K <= 0) || (q <= 0)) return 0.;
    if (q <= 4. * ELECTRON_MASS) return 0.;
    if (q >= K + q_offset(mass, PAIR_SQRTE, c)) return 0.;
    const double gamma = 1. + K / mass;
    const double x0 = 1. - 4. * ELECTRON_MASS / q;
    const double x1 = 1. - 6. / (gamma * (gamma - q / mass));
    if (!((x0 > 0) && (x1 > 0))) return 0.;
    const double rmax = sqrt(x0) * x1;
    const double ri = 1. - rmax;
    if ((ri <= 0.) || (ri >= 1.)) return 0.;
    const double tmin = fm::log_sel(ri, tb);
    // the DDCS's own range check (pumas.c:14469-14471) holds at every node:
    // 4 m_e < q < K + the offset
    const PairQ s = pair_setup(c, rl, mass, K, q, pair_zeta(c, mass, K, tb));
    double I = 0.;
#pragma unroll 1
    for (int i = 0; i < 12; i++) {
        const double rho = fm::exp(GQ12_X[i] * tmin, tb);
        I -= pair_d2_ssr(s, G, rho, tb) * rho * GQ12_W[i] * tmin;
    }
    return (I < 0) ? 0. : I;
}

// ALLM97 proton structure function F2 (pumas.c:14690-14745); lq0 is
// fm::log_sel(Q0^2 / Lambda^2, tb).
__device__ double f2p_allm97(double x, double Q2, double lq0, const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double m02 = 0.31985, mP2 = 49.457, mR2 = 0.15052, Q02 = 0.52544, Lambda2 = 0.06527;
    const double M2 = NUCLEON_MASS * NUCLEON_MASS;
    const double W2 = M2 + Q2 * (1.0 / x - 1.0);
    const double t = fm::log_sel(fm::log_sel((Q2 + Q02) / Lambda2, tb) / lq0, tb);
    // t^c as exp(c log t); t is 0 in exact arithmetic as Q2 -> 0, and clamped there
    const double lnt = fm::log_sel(t < 0. ? 0. : t, tb);
    const double xP = (Q2 + mP2) / (Q2 + mP2 + W2 - M2);
    const double xR = (Q2 + mR2) / (Q2 + mR2 + W2 - M2);
    const double cP = 0.28067 + (0.28067 - 0.22291) * (1.0 / (1.0 + fm::exp(2.1979 * lnt, tb)) - 1.0);
    const double aP = -0.0808 + (-0.0808 - -0.44812) * (1.0 / (1.0 + fm::exp(1.1709 * lnt, tb)) - 1.0);
    const double bP = 0.36292 + 1.8917 * fm::exp(1.8439 * lnt, tb);
    const double cR = 0.80107 + 0.97307 * fm::exp(3.4942 * lnt, tb);
    const double aR = 0.58400 + 0.37888 * fm::exp(2.6063 * lnt, tb);
    const double bR = 0.01147 + 3.7582 * fm::exp(0.49338 * lnt, tb);
    const double l1x = fm::log_sel(1 - x, tb);
    const double F2P = cP * fm::exp(aP * fm::log_sel(xP, tb) + bP * l1x, tb);
    const double F2R = cR * fm::exp(aR * fm::log_sel(xR, tb) + bR * l1x, tb);
    return Q2 / (Q2 + m02) * (F2P + F2R);
}

// DRSS photonuclear DDCS d2S / (dq dQ2) (pumas.c:14752-14785, 14987-15010).
__device__ double photo_d2_drss(const ElementConsts& c, const Globals& G, double ml, double K, double q, double Q2,
                                const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double Z = c.Z, A = c.A;
    const double cf = 4 * PI * ALPHA_EM * ALPHA_EM * HBAR_C * HBAR_C;
    const double E = K + ml;
    const double y = q / E;
    const double x = 0.5 * Q2 / (NUCLEON_MASS * q);
    const double F2p = f2p_allm97(x, Q2, G.lq0, tb);
    double shadowing;
    if (Z == 1.)
        shadowing = 1.;
    else if (x < 0.0014)
        shadowing = c.shadow_low;
    else if (x < 0.04)
        shadowing = fm::exp((0.069 * (fm::log_sel(x, tb) * INV_LN10) + 0.097) * c.lnA, tb);
    else
        shadowing = 1.;
    const double F2A = F2p * shadowing * (Z + (A - Z) * (1.0 + x * (-1.85 + x * (2.45 + x * (-2.35 + x)))));
    const double dds = (1 - y + 0.5 * (1 - 2 * ml * ml / Q2) * (y * y + Q2 / (E * E)) / (1 + 0.)) / (Q2 * Q2) -
                       0.25 / (E * E * Q2);
    return cf * F2A * dds / q;
}

// DRSS photonuclear, atomic DCS in m^2 / GeV (pumas.c:15066-15146, mode 0):
// the 9-point rule on ln Q^2 over [Q2min, Q2max].
__device__ double photo_drss(const ElementConsts& c, const Globals& G, double ml, double K, double q,
                             const fm::Tab& tb) {
#pragma clang fp contract(off)
    if ((c.Z <= 0) || (c.A <= 0) || (ml <= 0) || (K <= 0)) return 0.;
    const double M = NUCLEON_MASS;
    const double mpi = PION_MASS;
    if ((q <= mpi + 0.5 * mpi * mpi / M) || (q >= K + ml - 0.5 * (M + ml * ml / M))) return 0.;
    const double E = K + ml;
    const double ml2 = ml * ml;
    const double Q2min = ml2 * (q * q - 0.5 * ml2) / (E * (E - q));
    const double Q2max = 2.0 * M * (q - mpi) - mpi * mpi;
    if ((Q2max < Q2min) | (Q2min < 0)) return 0.;
    const double lmin = fm::log_sel(Q2min, tb);
    const double dx = fm::log_sel(Q2max, tb) - lmin;
    double ds = 0.;
#pragma unroll 1
    for (int i = 0; i < 9; i++) {
        const double Q2 = fm::exp(lmin + dx * GQ9_X[i], tb);
        const double tmp = photo_d2_drss(c, G, ml, K, q, Q2, tb);
        if (tmp <= 0.) continue;
        ds += tmp * (GQ9_W[i] * (dx * Q2));
    }
    return (ds < 0.) ? 0. : ds;
}

// Node `node` of pair_ssr's rule, with skip set where pair_ssr returns 0.
__device__ __forceinline__ void pair_term(const ElementConsts& c, double rl, const Globals& G, double mass, double K,
                                          double q, double zeta, int node, double* term, int* skip, const fm::Tab& tb) {
#pragma clang fp contract(off)
    if ((c.Z <= 0) || (c.A <= 0) || (mass <= 0) || (K <= 0) || (q <= 0)) return;
    if (q <= 4. * ELECTRON_MASS) return;
    if (q >= K + q_offset(mass, PAIR_SQRTE, c)) return;
    const double gamma = 1. + K / mass;
    const double x0 = 1. - 4. * ELECTRON_MASS / q;
    const double x1 = 1. - 6. / (gamma * (gamma - q / mass));
    if (!((x0 > 0) && (x1 > 0))) return;
    const double rmax = sqrt(x0) * x1;
    const double ri = 1. - rmax;
    if ((ri <= 0.) || (ri >= 1.)) return;
    const double tmin = fm::log_sel(ri, tb);
    const PairQ s = pair_setup(c, rl, mass, K, q, zeta);
    const double rho = fm::exp(GQ12_X[node] * tmin, tb);
    *term = pair_d2_ssr(s, G, rho, tb) * rho * GQ12_W[node] * tmin;
    *skip = 0;
}

// Node `node` of photo_drss's rule inside dcs()'s range, with skip set where
// the DCS is 0 or the node is left out of the sum.
__device__ __forceinline__ void photo_term(const ElementConsts& c, const Globals& G, double ml, double K, double q,
                                           int node, double* term, int* skip, const fm::Tab& tb) {
#pragma clang fp contract(off)
    const double M = NUCLEON_MASS;
    const double mpi = PION_MASS;
    if ((q < mpi + 0.5 * mpi * mpi / M) || (q > K + ml - 0.5 * (M + ml * ml / M))) return;
    if ((c.Z <= 0) || (c.A <= 0) || (ml <= 0) || (K <= 0)) return;
    if ((q <= mpi + 0.5 * mpi * mpi / M) || (q >= K + ml - 0.5 * (M + ml * ml / M))) return;
    const double E = K + ml;
    const double ml2 = ml * ml;
    const double Q2min = ml2 * (q * q - 0.5 * ml2) / (E * (E - q));
    const double Q2max = 2.0 * M * (q - mpi) - mpi * mpi;
    if ((Q2max < Q2min) | (Q2min < 0)) return;
    const double lmin = fm::log_sel(Q2min, tb);
    const double dx = fm::log_sel(Q2max, tb) - lmin;
    const double Q2 = fm::exp(lmin + dx * GQ9_X[node], tb);
    const double tmp = photo_d2_drss(c, G, ml, K, q, Q2, tb);
    *skip = tmp <= 0.;
    *term = tmp * (GQ9_W[node] * (dx * Q2));
}

// The m^2/kg DCS of process 0 (bremsstrahlung), 1 (pair production) or 2
// (photonuclear) as dcs_get(process) returns it (pumas.c:11018-11112).
__device__ double dcs(int process, const ElementConsts& c, const Globals& G, double mass, double K, double q,
                      const fm::Tab& tb) {
#pragma clang fp contract(off)
    double d;
    if (process == 0) {
        d = brems_ssr(c, rad_log(c.Z), G, mass, K, q, tb);
    } else if (process == 1) {
        d = pair_ssr(c, rad_log(c.Z), G, mass, K, q, tb);
    } else {
        const double qmin = PION_MASS + 0.5 * PION_MASS * PION_MASS / NUCLEON_MASS;
        const double qmax = K + mass - 0.5 * (NUCLEON_MASS + mass * mass / NUCLEON_MASS);
        if ((q < qmin) || (q > qmax)) return 0.;
        d = photo_drss(c, G, mass, K, q, tb);
    }
    return d * 1E+03 * AVOGADRO_NUMBER * (mass + K) / c.A;
}

__global__ __launch_bounds__(256) void pumas_dcs_kernel(int process, ElementConsts c, Globals G, double mass,
                                                        const double* __restrict__ K, const double* __restrict__ q,
                                                        int64_t n, double* __restrict__ out) {
    NOA_PUMAS_TABLES();
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        out[i] = dcs(process, c, G, mass, K[i], q[i], tb);
}

// Table row r = (p n_el + e0 + j) n_K + k: process, block element, energy. One
// workgroup holds as many rows of one (p, j) as its lanes have room for, a
// lane per node: the 36 nodes of a cutoff of 0.05 alone leave 28 of a wave's
// lanes idle. Bound: FP64 VALU, the nodes' quadratures run lane by lane.
// Measured for 48 elements x 146 energies: 158 us, a wave per row 290.
// Pair production's rows, the longest, start first.
constexpr int TABLE_WG = 256;
constexpr int TABLE_ROWS = TABLE_WG / N_REVERSE;  // a grid has at least N_REVERSE nodes

// A launch runs the call's workgroups from number `start` on.
__global__ __launch_bounds__(TABLE_WG) void pumas_table_kernel(Grid g, ElementBlock blk, Globals G, int64_t start,
                                                               int32_t e0, int32_t n_blk, int32_t n_el, double mass,
                                                               const double* __restrict__ Ks, int32_t n_K,
                                                               float* __restrict__ table, double* __restrict__ table64,
                                                               float* __restrict__ x_out, float* __restrict__ env,
                                                               const double* __restrict__ csn) {
#pragma clang fp contract(off)
    NOA_PUMAS_TABLES();
    __shared__ double xs[MAX_X];
    __shared__ double ys_all[TABLE_WG], ms_all[TABLE_WG];
    __shared__ int first[TABLE_ROWS], end[TABLE_ROWS], low[TABLE_ROWS], high[TABLE_ROWS];
    const int n = g.n;
    const int room = TABLE_WG / n;
    const int groups = (n_K + room - 1) / room;
    const int64_t b = start + blockIdx.x;
    const int p = int(b / (int64_t(n_blk) * groups) + 1) % 3;
    const int j = int((b / groups) % n_blk);
    const int row = int(threadIdx.x) / n, i = int(threadIdx.x) % n;
    const int k = int(b % groups) * room + row;
    const bool live = row < room && k < n_K;
    const int64_t r = (int64_t(p) * n_el + e0 + j) * n_K + k;
    const ElementConsts& c = blk.e[j];
    if (threadIdx.x < unsigned(n)) {
        xs[threadIdx.x] = g.x[threadIdx.x];
        if (b == 0 && x_out) x_out[threadIdx.x] = float(g.x[threadIdx.x]);
    }
    if (threadIdx.x < TABLE_ROWS) {
        first[threadIdx.x] = end[threadIdx.x] = n;
        low[threadIdx.x] = n;
        high[threadIdx.x] = -1;
    }
    __syncthreads();
    // no cross section: an empty row (pumas.c:11427-11434)
    const bool some = live && !(csn && !(csn[r] > 0.));
    double* ys = ys_all + (live ? row * n : 0);
    double* ms = ms_all + (live ? row * n : 0);
    const double K = live ? Ks[k] : 1.;
    bool positive = false;
    if (some) {
        const double q = K * fm::exp(xs[i], tb);
        const double d = dcs(p, c, G, mass, K, q, tb);
        positive = d > 0;
        ys[i] = positive ? fm::log_sel(d, tb) : 0.;
        if (positive) atomicMin(&first[row], i);
    }
    __syncthreads();
    // the first run of positive values
    const int imin = some ? first[row] : n;
    if (some && !positive && i > imin) atomicMin(&end[row], i);
    __syncthreads();
    const int imax = (some ? end[row] : n) - 1;
    // PCHIP slopes over [imin, imax] (math_pchip_initialise with der = 0)
    const int N = imax - imin + 1;
    if (some) {
        double m = 0.;
        if (N >= 1 && i >= imin && i <= imax) {
            const double* x = xs + imin;
            const double* y = ys + imin;
            int j = i - imin;
            int nn = N;
            if (N >= 3) {
                if (j == 0) {
                    m = (y[1] - y[0]) / (x[1] - x[0]);
                    goto done;
                }
                x++;
                y++;
                j--;
                nn--;
            }
            if (nn == 1) {
                m = 0.;
            } else if (nn == 2) {
                m = (y[1] - y[0]) / (x[1] - x[0]);
            } else if (j == 0 || j == nn - 1) {
                // three-point end derivative (math_diff3, pumas.c:10010-10020)
                const int a = j, b = (j == 0) ? 1 : nn - 2, c = (j == 0) ? 2 : nn - 3;
                const double h1 = x[b] - x[a];
                const double h2 = x[c] - x[a];
                const double delta = h1 * h2 * (h2 - h1);
                const double c1 = h2 * h2 / delta;
                const double c2 = -h1 * h1 / delta;
                const double c0 = -(c1 + c2);
                m = c0 * y[a] + c1 * y[b] + c2 * y[c];
            } else {
                const double h1 = x[j] - x[j - 1];
                const double h2 = x[j + 1] - x[j];
                const double S1 = (y[j] - y[j - 1]) / h1;
                const double S2 = (y[j + 1] - y[j]) / h2;
                const double tmp = S1 * S2;
                if (tmp > 0) {
                    const double a = (h1 + 2 * h2) / (3 * (h1 + h2));
                    m = tmp / ((1 - a) * S1 + a * S2);
                } else {
                    m = 0.;
                }
            }
        }
    done:
        ms[i] = m;
        const bool in = i >= imin && i <= imax;
        float* out = table + r * 2 * n;
        out[2 * i] = in ? float(ys[i]) : 0.f;
        out[2 * i + 1] = in ? float(m) : 0.f;
        if (table64) {
            double* out64 = table64 + r * 2 * n;
            out64[2 * i] = in ? ys[i] : 0.;
            out64[2 * i + 1] = in ? m : 0.;
        }
        if (env && in) {
            // the nodes of the envelope exponent's range (pumas.c:11462-11507)
            double qmin, qmax;
            if (p == 2) {
                qmin = PION_MASS + 0.5 * PION_MASS * PION_MASS / NUCLEON_MASS;
                qmax = K + mass - 0.5 * (NUCLEON_MASS + mass * mass / NUCLEON_MASS);
                qmin += qmin;
            } else {
                qmax = K + q_offset(mass, PAIR_SQRTE, c);
                qmin = (p == 0) ? 0.5 * g.cutoff * K : 4. * ELECTRON_MASS * 4;
            }
            const double qrev = X_REVERSE * K;
            qmax *= 0.5;
            if (qmax > qrev) qmax = qrev;
            if ((xs[i] > fm::log_sel(qmin / K, tb)) && (xs[i] < fm::log_sel(qmax / K, tb))) {
                atomicMin(&low[row], i);
                atomicMax(&high[row], i);
            }
        }
    } else if (live) {
        float* out = table + r * 2 * n;
        out[2 * i] = out[2 * i + 1] = 0.f;
        if (table64) {
            double* out64 = table64 + r * 2 * n;
            out64[2 * i] = out64[2 * i + 1] = 0.;
        }
    }
    __syncthreads();
    if (live && i == 0 && env) {
        float alpha = 0.f;  // an empty row: the reference leaves the pair as it was; here 0
        if (some) {
            const int ia0 = min(imax, low[row]), ia1 = max(imin, high[row]);
            if ((ia0 < ia1) && (ia0 < n - 1)) {
                const int ia = (3 * ia0 + ia1) / 4;
                double a = -ms[ia];
                if (fabs(a - 1.) <= 0.1) a = 1.;
                alpha = float(a);
            }
        }
        env[2 * r] = alpha;
        env[2 * r + 1] = 0.f;
    }
}

// Rows below the first positive envelope exponent of a (process, element)
// take that exponent (pumas.c:11745-11761). One wave per (process, element).
__global__ __launch_bounds__(64) void pumas_alpha_fill_kernel(float* __restrict__ env, int32_t n_K) {
    float* a = env + 2 * int64_t(blockIdx.x) * n_K;
    const int lane = threadIdx.x;
    for (int row = 0; row < n_K; row += 64) {
        const float v = row + lane < n_K ? a[2 * int64_t(row + lane)] : 0.f;
        const unsigned long long positive = __ballot(v > 0.f);
        if (!positive) continue;
        const int at = __ffsll((long long)positive) - 1;
        const float alpha = __shfl(v, at, 64);
        for (int below = lane; below < row + at; below += 64) a[2 * int64_t(below)] = alpha;
        return;
    }
}

// The quadrature nodes of up to this many model evaluations fill one wave:
// 5 x 12 (pair production), 7 x 9 (photonuclear); bremsstrahlung has no nodes.
__device__ __forceinline__ int model_batch(int process) { return process == 0 ? 64 : process == 1 ? 5 : 7; }

// What a lane pushed to this one (several to one lane: one of them; none: 0).
__device__ __forceinline__ double push_to(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = uint32_t(__builtin_amdgcn_ds_permute(4 * lane, int(uint32_t(u))));
    const uint32_t hi = uint32_t(__builtin_amdgcn_ds_permute(4 * lane, int(uint32_t(u >> 32))));
    return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// The m^2/kg model DCS of one (K, q) per lane, for the lanes with need set (K
// the same in every lane; the other lanes get 0). A wave takes model_batch
// evaluations at a time, a group of lanes each: every lane of a group forms
// the set-up and one quadrature node, and the node terms are summed in the
// serial loop's order, so the values are those of dcs() bit for bit. Must be
// called with the wave's 64 lanes active.
__device__ __forceinline__ double dcs_wave(int process, const ElementConsts& c, double rl, const Globals& G, double mass,
                                           double K, double zeta, double q, bool need, const fm::Tab& tb) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63;
    double d = 0.;
    if (process == 0) {
        if (need) d = brems_ssr(c, rl, G, mass, K, q, tb);
    } else {
        const int nodes = process == 1 ? 12 : 9;
        const int per = model_batch(process);
        const int group = lane / nodes, node = lane - group * nodes;
        const unsigned long long todo = __ballot(need);
        const int total = __popcll(todo);
        const int rank = __popcll(todo & ((1ull << lane) - 1));
        for (int base = 0; base < total; base += per) {
            // the group's evaluation is that of the group-th lane still to do,
            // which hands its q to lane `group`
            const int mine = rank - base;
            const int owner_group = need && mine >= 0 && mine < per ? mine : -1;
            const double qg = __shfl(push_to(q, owner_group < 0 ? 63 : owner_group), group, 64);
            double term = 0.;
            int skip = 1;
            if (group < min(per, total - base)) {
                if (process == 1)
                    pair_term(c, rl, G, mass, K, qg, zeta, node, &term, &skip, tb);
                else
                    photo_term(c, G, mass, K, qg, node, &term, &skip, tb);
            }
            const int first = (owner_group < 0 ? 0 : owner_group) * nodes;
            double sum = 0.;
            if (process == 1) {
                const int skipped = __shfl(skip, first, 64);  // a whole evaluation at once
#pragma unroll
                for (int i = 0; i < 12; i++) sum -= __shfl(term, first + i, 64);
                if (skipped) sum = 0.;
            } else {
                if (skip) term = 0.;
#pragma unroll
                for (int i = 0; i < 9; i++) sum += __shfl(term, first + i, 64);
            }
            if (owner_group >= 0) d = (sum < 0) ? 0. : sum;
        }
    }
    return need ? d * 1E+03 * AVOGADRO_NUMBER * (mass + K) / c.A : 0.;
}

// ---- the envelope maximum (dcs_tabulate_envelope_row, pumas.c:11526-11679) ----
//
// One wave per row. The reference searches the maximum of DCS x^alpha over ln x
// serially, 100 to 240 evaluations of one point each: bisections that find
// where the DCS becomes positive at the range ends, then two bracketing
// bisections, one in each half of the range (math_find_minimum with algo 0,
// pumas.c:12172-12232 and 12416-12459), and for pair production at K >= 1e7 a
// logarithmic scan next to the upper end. DCS is the table interpolated as
// dcs_evaluate does without a context (pumas.c:11307-11398) and the model
// where the table does not apply. The rows read are those of the finished
// table.
//
// Every step of those searches has two outcomes and the next point depends
// only on the outcomes so far, so half a wave evaluates the points of a
// search's next 5 steps at once, all 31 of their decision tree, one per lane,
// and then walks the tree: the points and decisions of the serial search. The
// two halves run the two bracketing searches side by side. Where points need
// the model, fewer steps: as many as their model evaluations fit one batch of
// dcs_wave (5 of pair production, 7 of photonuclear).
//
// Where the range end is the logarithm of a negative number (K below the
// kinematic threshold) the reference's search makes 200 evaluations at NaN;
// they all have the first one's value, so two evaluations settle the row.
//
// The reference's search reads the nodes from physics->table_DCS_x, which
// compute_dcs_table writes only after element 0 (pumas.c:11775-11783), so
// element 0's search sees zero nodes and takes the model everywhere; the
// kernel does the same.
//
// What bounds it is the instructions of a row's chain of rounds (about 20, up
// to 60 where every point needs the model, of ~500 to 2000 vector instructions
// each), with three waves per SIMD to overlap: the vector units are busy 73% of
// the launch. Measured for 48 elements x 146 energies, the whole table call:
// one point per step for the whole wave 10,600 us; trees of one search per wave
// 4113; two searches side by side with the table log / exp 2810; the rows'
// constants and the searches kept out of the registers 1980; one launch for 48
// elements 1334; a tree's nodes taking their steps at once 1217; selections for
// branches 1177; model batches filled point by point 1105; a copy of the search
// per process, the longest rows first and the logarithms without branches 953.

// v of one lane, as a wave-uniform (scalar) value.
__device__ __forceinline__ double from_lane(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const int l = __builtin_amdgcn_readfirstlane(lane);
    const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u)), l));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u >> 32)), l));
    return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

struct EnvRow {
    int process;
    double mass;
    double rl;          // rad_log(Z)
    const float* xt;    // the nodes as the search sees them (LDS)
    int n;
    // dcs_evaluate's energy bracket: K is the row's own energy at every
    // evaluation, so the two rows it reads (LDS copies) and their weights
    // are fixed per row
    const float* ra;  // row i0 (or the last row)
    const float* rb;  // row i0 + 1 (or the last row again)
    float h0, h1;
    double qmin, qlow, qmax;  // table_range
    bool below;  // K below the grid (never the case for a row's own energy)
};

// table_index without a context (pumas.c:4249-4290, 4299-4306).
__device__ __forceinline__ int table_index(const double* table, int n_K, double value) {
    const int imax = n_K - 1;
    if (value < table[0]) return -1;
    if (value >= table[imax]) return imax;
    int i1 = 0, i2 = imax;
    while (true) {
        const int i3 = (i1 + i2) / 2;
        if (value >= table[i3])
            i1 = i3;
        else
            i2 = i3;
        if (i2 - i1 < 2) break;
    }
    return i1;
}

// The range of dcs_evaluate (pumas.c:11319-11349): 0 outside [qmin, qmax], the
// model below qlow.
__device__ __forceinline__ void table_range(EnvRow& a, const ElementConsts& c, double K) {
#pragma clang fp contract(off)
    if (a.process == 2) {
        a.qmin = PION_MASS + 0.5 * PION_MASS * PION_MASS / NUCLEON_MASS;
        a.qmax = K + a.mass - 0.5 * (NUCLEON_MASS + a.mass * a.mass / NUCLEON_MASS);
        a.qlow = 2 * a.qmin;
    } else {
        a.qmin = a.process == 1 ? 4. * ELECTRON_MASS : 0.;
        a.qmax = K + q_offset(a.mass, PAIR_SQRTE, c);
        a.qlow = 4 * a.qmin;
    }
    a.qmax = from_lane(a.qmax, 0);
}

// The interpolated DCS at q without its factor K / (K + m), or *need set where
// it is the model's. Without early returns: a wave's lanes rarely differ in
// them, and each cost a branch.
__device__ __forceinline__ double dcs_from_table(const EnvRow& a, double K, double q, bool* need) {
#pragma clang fp contract(off)
    const bool in = !((q < a.qmin) || (q > a.qmax));
    const int nx = a.n;
    const float x = logf((float)(q / K));
    bool ok = in && !(q < a.qlow) && !((x < a.xt[0]) || (x >= a.xt[nx - 1])) && !a.below;
    float r = 0.f;
    if (__ballot(ok)) {
        const int ix = cell(a.xt, nx, x, ok);
        const float p00 = a.ra[2 * ix], p01 = a.ra[2 * ix + 2], p10 = a.rb[2 * ix], p11 = a.rb[2 * ix + 2];
        float m00 = a.ra[2 * ix + 1], m01 = a.ra[2 * ix + 3], m10 = a.rb[2 * ix + 1], m11 = a.rb[2 * ix + 3];
        ok = ok & !(((p00 == 0.f) & (m00 == 0.f)) | ((p01 == 0.f) & (m01 == 0.f)) | ((p10 == 0.f) & (m10 == 0.f)) |
                    ((p11 == 0.f) & (m11 == 0.f)));
        const float x0 = a.xt[ix];
        const float x1 = a.xt[ix + 1];
        const float dx = x1 - x0;
        m00 *= dx;
        m01 *= dx;
        const float t = (x - x0) / dx;
        const float c02 = -3 * (p00 - p01) - 2 * m00 - m01;
        const float c03 = 2 * (p00 - p01) + m00 + m01;
        r = expf(p00 + t * (m00 + t * (c02 + t * c03))) * a.h0;
        if (a.h1 > 0.f) {
            m10 *= dx;
            m11 *= dx;
            const float c12 = -3 * (p10 - p11) - 2 * m10 - m11;
            const float c13 = 2 * (p10 - p11) + m10 + m11;
            r += expf(p10 + t * (m10 + t * (c12 + t * c13))) * a.h1;
        }
    }
    *need = in && !ok;
    return ok ? r : 0.f;
}

// One search of a half-wave, or its state at one node of the decision tree.
enum SearchKind { SEARCH_NONE, SEARCH_EDGE, SEARCH_BRACKET, SEARCH_BISECT };
constexpr double RESOLUTION = 1E-10;

struct Search {
    int kind;
    // EDGE: bisection of [xa, xc] for the edge of the region where f != 0; the
    //   nonzero side is xc (up) or xa; xb, fb the last nonzero point and value
    // BRACKET: find_minimum's first stage, halving [xa, xc] towards the lower
    //   end until the midpoint lies below both ends
    // BISECT: find_minimum's bisection around xb; fb is the result
    double xa, xb, xc, fa, fb, fc, tol;
    int i, max_iter, up;

    __device__ __forceinline__ bool done() const {
        if (kind == SEARCH_EDGE) return !(xc - xa > RESOLUTION);
        if (kind == SEARCH_BISECT) return !((xc - xa > tol) && (i < max_iter));
        return kind == SEARCH_NONE;
    }
    __device__ __forceinline__ double point() const {
        const bool low = kind != SEARCH_BISECT || xb - xa > xc - xb;
        const double u = (kind == SEARCH_BISECT && !low) ? xb : xa;
        const double v = (kind == SEARCH_BISECT && low) ? xb : xc;
        return 0.5 * (u + v);
    }
    // The state's points after outcome `bit` of the next step. EDGE: 1 =
    // nonzero; BRACKET: 1 = the minimum is right; BISECT: 1 = lower than xb.
    __device__ __forceinline__ void next(int bit) {
        const double x = point();
        if (kind == SEARCH_BISECT) {
            const bool low = xb - xa > xc - xb;
            const double b = xb;
            if (bit) xb = x;
            // lower on the low side: xc = old xb; on the high side: xa = old
            // xb; not lower: the bracket's end on that side moves to x
            if (low == bool(bit))
                xc = bit ? b : x;
            else
                xa = bit ? b : x;
        } else {
            const bool to_c = kind == SEARCH_EDGE ? bit == up : !bit;
            if (kind == SEARCH_EDGE && bit) xb = x;
            if (to_c)
                xc = x;
            else
                xa = x;
        }
    }
    // The true step with value v at point(): its outcome, or -1 where the
    // tree ends with it.
    __device__ __forceinline__ int step(double v) {
        int bit;
        if (kind == SEARCH_EDGE) {
            bit = v != 0;
            if (bit) fb = v;
        } else if (kind == SEARCH_BISECT) {
            bit = v < fb;
            if (bit) fb = v;
            i++;
        } else {  // BRACKET
            xb = point();
            fb = v;
            if ((fb < fa) && (fb < fc)) {  // bracketed: on to the bisection, with the iterations left
                kind = SEARCH_BISECT;
                tol = RESOLUTION * fabs(xc - xa);
                max_iter -= i;
                i = 0;
                return -1;
            }
            i++;
            if (fabs(xc - xa) <= tol) {  // spent
                kind = SEARCH_NONE;
                return -1;
            }
            bit = !(fb < fc);
            if (bit)
                fa = fb;
            else
                fc = fb;
            next(bit);
            if (i >= max_iter) {
                kind = SEARCH_NONE;
                if (fa < fb)
                    fb = fa;
                else if (fc < fb)
                    fb = fc;
                return -1;
            }
            return bit;
        }
        next(bit);
        return bit;
    }
};

__device__ __forceinline__ Search new_search(int kind, double xa, double xc, double fa, double fc, double tol, int up,
                                             double xb, double fb) {
    Search s;
    s.kind = kind;
    s.xa = xa;
    s.xb = xb;
    s.xc = xc;
    s.fa = fa;
    s.fb = fb;
    s.fc = fc;
    s.tol = tol;
    s.i = 0;
    s.max_iter = 100;
    s.up = up;
    return s;
}

// Orders the wave's LDS accesses before and after it.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Stores a half's search (its 32 lanes hold the same values).
__device__ __forceinline__ void put(Search& to, const Search& s) {
    wave_lds_order();
    to = s;
    wave_lds_order();
}

// The row's constants in the kernel-argument segment, re-read where they are
// used: an empty asm hides the pointer, and hide() a value, so that what
// follows from them alone is not formed before the search and held in
// registers throughout (it took 250 VGPRs, two waves per SIMD).
using ElementPtr = const __attribute__((address_space(4))) ElementConsts*;
__device__ __forceinline__ const ElementConsts& row_consts(ElementPtr p) {
    asm volatile("" : "+s"(p));
    return *(const ElementConsts*)p;
}
__device__ __forceinline__ double hide(double v) {
    asm volatile("" : "+s"(v));
    return v;
}

template <int Process>
__device__ __forceinline__ float envelope_max(const EnvRow& a, ElementPtr cp, const Globals& G, double K, double cutoff,
                                               float alpha_f, double cs, Search* searches, double (*tree)[64],
                                               const fm::Tab& tb) {
#pragma clang fp contract(off)
    const ElementConsts& c0 = *(const ElementConsts*)cp;
    const int lane = threadIdx.x & 63;
    const int half = lane >> 5, node = lane & 31;
    // the tree's nodes are numbered by level (children 2 node + 1 + outcome):
    // node + 1 in binary is a one and the outcomes on the path to the node.
    // last1, last0: the last node on that path with outcome 1 and 0, or -1
    const int depth = 31 - __clz(node + 1);
    const int last1 = ((node + 1) >> __ffs(node + 1)) - 1;
    const int last0 = ((node + 1) >> __ffs(~(node + 1))) - 1;
    if (cs <= 0.) return 0.f;
    const double alpha = (double)alpha_f;
    double qmin, qmax;
    if (Process == 2) {  // dcs_get_range (pumas.c:11047-11056)
        qmin = PION_MASS + 0.5 * PION_MASS * PION_MASS / NUCLEON_MASS;
        qmax = K + a.mass - 0.5 * (NUCLEON_MASS + a.mass * a.mass / NUCLEON_MASS);
    } else {
        qmin = (Process == 0) ? 0. : 4. * ELECTRON_MASS;
        qmax = K + q_offset(a.mass, PAIR_SQRTE, c0);
    }
    double xmin = qmin / K;
    if (xmin < cutoff) xmin = cutoff;
    xmin = fm::log_sel(xmin, tb);
    double xmax = fm::log_sel(qmax / K, tb);
    if (xmin >= xmax) return 0.f;
    const double wj = K / (K + a.mass);
    const int batch = model_batch(Process);
    const double zeta = Process == 1 ? pair_zeta(c0, a.mass, K, tb) : 0.;

    // ENDS: the range ends and the midpoint; EDGE_LOW, BACKOFF, EDGE_HIGH: the
    // ends' searches; MID: the midpoint between moved ends; PAIR: the two
    // bracketing searches; SCAN and PEAK: the scan next to the upper end
    enum { ENDS, EDGE_LOW, BACKOFF, EDGE_HIGH, MID, PAIR, SCAN, PEAK } phase = ENDS;
    constexpr int N_SCAN = 7;
    // the halves' searches live in LDS: not in registers across an evaluation
    Search& s = searches[half];
    double f0 = 0., f1 = 0., fmid = 0., fopt0 = 0., fopt1 = 0.;
    double delta = RESOLUTION, exm = 0.;
    bool moved = false;
#pragma unroll 1
    for (;;) {
        const ElementConsts& c = row_consts(cp);
        const double mass = hide(a.mass);
        // this lane's point, and whether it is part of a tree or one of n points
        double lnx;
        int points = 0;
        if (phase == ENDS) {
            points = 3;
            lnx = lane == 0 ? xmin : lane == 1 ? xmax : 0.5 * (xmin + xmax);
        } else if (phase == MID) {
            points = 1;
            lnx = 0.5 * (xmin + xmax);
        } else if (phase == BACKOFF) {
            points = batch;
            lnx = fm::log_sel(exm - ldexp(delta, lane < points ? lane : 0), tb);
        } else if (phase == SCAN) {
            points = N_SCAN;
            // xmax + log(1 - 10^-(i + 1))
            lnx = xmax + fm::log_sel(1. - pow(10., double(-((lane < N_SCAN ? lane : 0) + 1))), tb);
        } else {
            // the search's state at this lane's node
            wave_lds_order();
            Search mine = s;
#pragma unroll 1
            for (int l = 3; l >= 0; l--)
                if (l < depth && node < 31) mine.next((node + 1) >> l & 1);
            lnx = mine.point();
            tree[0][lane] = mine.xa;
            tree[1][lane] = mine.xb;
            tree[2][lane] = mine.xc;
        }
        // -DCS x^alpha there
        const double x = fm::exp(lnx, tb);
        const double q = x * K;
        bool need;
        double d = dcs_from_table(a, K, q, &need);
        const bool asked = need;
        if (points) {
            need = need && lane < points;
        } else {
            need = need && !s.done() && node < 31;
            const unsigned long long m = __ballot(need);
            if (m) {
                // the model's points in the order of their levels, half 1 before
                // half 0, as many as one batch takes
                const uint32_t own = uint32_t(m >> (32 * half)), other = uint32_t(m >> (32 * (half ^ 1)));
                const int before = __popc(own & ((1u << node) - 1)) + __popc(other & tree_levels(depth + 1 - half));
                need = need && before < batch;
            }
        }
        if (__ballot(need)) {
            const double md = dcs_wave(Process, c, a.rl, G, mass, K, zeta, q, need, tb);
            if (need) d = md;
        }
        const double v = -(d * wj) * (alpha == 0. ? 1. : fm::exp(alpha * lnx, tb));

        if (!points) {
            // every node's own step, then the path through the outcomes; the
            // last node on it holds the search's new state
            const double up = __shfl(v, 32 * half + (last1 < 0 ? 0 : last1), 64);
            const double down = __shfl(v, 32 * half + (last0 < 0 ? 0 : last0), 64);
            Search mine = s;
            mine.xa = tree[0][lane];
            mine.xb = tree[1][lane];
            mine.xc = tree[2][lane];
            mine.i += depth;
            if (last1 >= 0) {
                mine.fa = up;
                if (mine.kind != SEARCH_BRACKET) mine.fb = up;
            }
            if (last0 >= 0) mine.fc = down;
            const bool go = (need || !asked) && node < 31 && !mine.done();
            const int bit = go ? mine.step(v) : -1;
            const uint32_t goes = uint32_t(__ballot(go) >> (32 * half));
            const uint32_t ends = uint32_t(__ballot(bit < 0) >> (32 * half));
            const uint32_t ones = uint32_t(__ballot(bit > 0) >> (32 * half));
            int at = 0, last = -1;
#pragma unroll
            for (int l = 0; l < 5; l++) {
                if (at < 31 && (goes >> at & 1)) {
                    last = at;
                    at = (ends >> at & 1) ? 31 : 2 * at + 1 + int(ones >> at & 1);
                } else {
                    at = 31;
                }
            }
            wave_lds_order();
            if (node == last) s = mine;
            wave_lds_order();
        }

        // what comes next (the same in every lane): `settled` counts the
        // parts that are complete, the lower end, the upper end, the midpoint
        // and the two searches
        int settled = 0;
        if (phase == ENDS) {
            f0 = from_lane(v, 0);
            f1 = from_lane(v, 1);
            fmid = from_lane(v, 2);
            if (xmax != xmax) {
                const double fopt = f0 < f1 ? f0 : f1;
                return (float)(-fopt);
            }
            if (f0 == 0.) {
                moved = true;
                put(s, new_search(half ? SEARCH_NONE : SEARCH_EDGE, xmin, xmax, 0., 0., 0., 1, xmin, f0));
                phase = EDGE_LOW;
            } else {
                settled = 1;
            }
        } else if (phase == BACKOFF) {
            // the first of exm - delta, delta = 1e-10 2^i, with f != 0
            const unsigned long long in = __ballot(lane < points && exm > ldexp(delta, lane < points ? lane : 0));
            const unsigned long long nz = __ballot(v != 0.) & in;
            const int i = nz ? __ffsll((long long)nz) - 1 : 63 - __clzll((long long)in);
            xmax = from_lane(lnx, i);
            f1 = from_lane(v, i);
            delta = ldexp(delta, nz ? i : i + 1);
            if (!nz && exm > delta) continue;
            put(s, new_search(half ? SEARCH_NONE : SEARCH_EDGE, xmax, fm::log_sel(exm - delta / 2, tb), 0., 0., 0., 0, xmax, f1));
            phase = EDGE_HIGH;
        } else if (phase == MID) {
            fmid = from_lane(v, 0);
            settled = 3;
        } else if (phase == SCAN) {
            double fmin = 0.;
            int imin = -1;
            for (int i = 0; i < N_SCAN; i++) {
                const double fi = from_lane(v, i);
                if (fi < fmin) {
                    imin = i;
                    fmin = fi;
                }
            }
            if (!((imin > 0) && (imin < N_SCAN - 1))) break;
            const double xa = from_lane(lnx, imin - 1), xc = from_lane(lnx, imin + 1);
            put(s, new_search(half ? SEARCH_NONE : SEARCH_BISECT, xa, xc, 0., 0., RESOLUTION * fabs(xc - xa), 0, from_lane(lnx, imin), fmin));
            phase = PEAK;
        }
        if (settled == 0) {  // a search is under way
            if (__ballot(!s.done())) continue;
            const double xs = from_lane(s.xb, 0), fs = from_lane(s.fb, 0);
            if (phase == EDGE_LOW) {
                xmin = xs;
                f0 = fs;
                settled = 1;
            } else if (phase == EDGE_HIGH) {
                xmax = xs;
                f1 = fs;
                settled = 2;
            } else if (phase == PAIR) {
                fopt0 = fs;
                fopt1 = from_lane(s.fb, 32);
                settled = 4;
            } else {  // PEAK
                if (fs < fopt1) fopt1 = fs;
                break;
            }
        }
        if (settled == 1) {
            if (f1 == 0.) {
                moved = true;
                if (K >= 1E+01) {
                    exm = fm::exp(xmax, tb);
                    phase = BACKOFF;
                    if (exm > delta) continue;
                }
                put(s, new_search(half ? SEARCH_NONE : SEARCH_EDGE, K >= 1E+01 ? xmax : xmin, K >= 1E+01 ? fm::log_sel(exm - delta / 2, tb) : xmax, 0., 0.,
                        0., 0, xmax, f1));
                phase = EDGE_HIGH;
                if (__ballot(!s.done())) continue;
            }
            settled = 2;
        }
        if (settled == 2) {
            phase = MID;
            if (moved) continue;
            settled = 3;
        }
        if (settled == 3) {
            const double xm = 0.5 * (xmin + xmax);
            const double lo = half ? xm : xmin, hi = half ? xmax : xm;
            put(s, new_search(SEARCH_BRACKET, lo, hi, half ? fmid : f0, half ? f1 : fmid, RESOLUTION * fabs(hi - lo), 0, xm,
                              fmid));
            phase = PAIR;
            continue;
        }
        if (!((Process == 1) && (K >= 1E+07))) break;
        phase = SCAN;
    }
    double fopt = (fopt0 < fopt1) ? fopt0 : fopt1;
    if (f0 < fopt) fopt = f0;
    if (f1 < fopt) fopt = f1;
    return (float)(-fopt);
}

// The leading arguments of pumas_envelope_kernel, as the kernel-argument
// segment holds them.
struct EnvelopeArgs {
    EnvelopeGrid g;
    EnvelopeBlock blk;
    Globals G;
    int32_t n_x, e0, n_blk, n_el;
    double mass, cutoff;
    const double* Ks;
    const float* table;
    const double* csn;
    float* env;
    int64_t start;  // number of the launch's first workgroup among the call's
    int32_t n_K;
};
static_assert(sizeof(EnvelopeArgs) <= MAX_KERNARG, "48 elements and the grid in one launch");

// The row's nodes and the two table rows it reads. (Sized by the grid, not by
// MAX_X: the LDS then holds 12 workgroups per CU, three waves per SIMD, up to
// ~145 nodes.)
constexpr int ENVELOPE_LDS = 5;

// One 64-lane workgroup per (process, block element j, kinetic energy k) row
// of the launch's element block; env[2 r + 1] of table row r. Rows start
// longest first: the first element's (element 0 takes the model at every
// point), then pair production's, and of each the lowest energies first: those
// just above the threshold, with few valid table nodes, take 2 to 3 times as
// long as the highest. The launch's length over its rows' sum is 1.20 with the
// highest energies first and 1.10 so (1095 against 1020 us for 48 elements x
// 146 energies).
template <int WAVES>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES))) void pumas_envelope_kernel(EnvelopeArgs by_value) {
    extern __shared__ float row_lds[];  // ENVELOPE_LDS floats per grid node
    __shared__ Search searches[2];
    __shared__ double tree[3][64];
    NOA_PUMAS_TABLES();
    const auto args = (const __attribute__((address_space(4))) EnvelopeArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    const Globals G = *(const Globals*)&args->G;
    const int32_t n_K = args->n_K, n_el = args->n_el, n_blk = args->n_blk, e0 = args->e0, n_x = args->n_x;
    float* const xt = row_lds;
    float* const ra = xt + n_x;
    float* const rb = ra + 2 * n_x;
    const double mass = args->mass;
    const double* __restrict__ Ks = args->Ks;
    const float* __restrict__ table = args->table;
    const double* __restrict__ csn = args->csn;
    float* __restrict__ env = args->env;
    int64_t b = args->start + blockIdx.x;
    int p = 1, j = 0;
    if (b < int64_t(3) * n_K) {
        p += int(b / n_K);
        b %= n_K;
    } else {
        b -= int64_t(3) * n_K;
        const int64_t rest = int64_t(n_blk - 1) * n_K;
        p += int(b / rest);
        b %= rest;
        j = 1 + int(b % (n_blk - 1));
        b /= n_blk - 1;
    }
    p %= 3;
    const int k = int(b);
    const int e = e0 + j;
    const int64_t pe = int64_t(p) * n_el + e;
    const int64_t r = pe * n_K + k;
    for (int i = threadIdx.x; i < n_x; i += 64) {
#pragma clang fp contract(off)
        const int m = args->g.m;
        const float x = i < m ? float(args->g.x0 + i * args->g.dx) : args->g.tail[i - m];
        xt[i] = (e == 0) ? 0.f : x;
    }
    // dcs_evaluate's energy bracket of the row's own energy (pumas.c:11352-11381)
    const double K = Ks[k];
    const float* rows = table + pe * n_K * 2 * n_x;
    const int imax = n_K - 1;
    int i0 = 0, ia = imax, ib = imax;
    float h0 = 1.f, h1 = 0.f;
    if (!((K >= Ks[imax]) || ((i0 = table_index(Ks, n_K, K)) >= imax)) && i0 >= 0) {
        ia = i0;
        ib = i0 + 1;
        const float K0 = (float)Ks[i0];
        const float K1 = (float)Ks[i0 + 1];
        h1 = logf(((float)K) / K0) / logf(K1 / K0);
        h0 = 1.f - h1;
    }
    for (int i = threadIdx.x; i < 2 * n_x; i += 64) {
        ra[i] = rows[int64_t(ia) * 2 * n_x + i];
        rb[i] = rows[int64_t(ib) * 2 * n_x + i];
    }
    __syncthreads();
    EnvRow a;
    a.process = p;
    a.mass = mass;
    a.n = n_x;
    a.xt = xt;
    a.ra = ra;
    a.rb = rb;
    a.h0 = h0;
    a.h1 = h1;
    a.below = i0 < 0;
    const ElementPtr cp = &args->blk.e[j];
    a.rl = rad_log(cp->Z);
    table_range(a, *(const ElementConsts*)cp, K);
    const float alpha = env[2 * r];
    const double cs = csn ? csn[r] : 1.;
    const float v = p == 0   ? envelope_max<0>(a, cp, G, K, args->cutoff, alpha, cs, searches, tree, tb)
                    : p == 1 ? envelope_max<1>(a, cp, G, K, args->cutoff, alpha, cs, searches, tree, tb)
                             : envelope_max<2>(a, cp, G, K, args->cutoff, alpha, cs, searches, tree, tb);
    if (threadIdx.x == 0) env[2 * r + 1] = v;
}

// The grid (pumas.c:1548-1554, 11712-11737), on the host with its libm.
inline int n_table(double cutoff) {
    int n = N_REVERSE;
    if (cutoff < X_REVERSE) {
        int m = int(std::log10(X_REVERSE / cutoff) * PER_DECADE);
        if (m < N_MIN) m = N_MIN;
        n += m;
    }
    return n;
}

inline Globals make_globals() {
#pragma clang fp contract(off)
    Globals G;
    G.e1 = std::exp(1.);
    G.e05 = std::exp(0.5);
    G.e_16 = std::exp(-1. / 6.);
    G.e13 = std::exp(1. / 3.);
    G.e_13 = std::exp(-1. / 3.);
    G.lq0 = std::log(0.52544 / 0.06527);
    return G;
}

// The element's launch invariants, each in the reference's expression and
// order (pumas.c:13985-14016, 14301, 14478-14481, 14760, 14632-14634).
inline ElementConsts make_element(double Z, double A, double mass, const Globals& G) {
#pragma clang fp contract(off)
    ElementConsts c;
    c.Z = Z;
    c.A = A;
    c.z13 = std::pow(Z, 1. / 3.);
    c.Z13m = std::pow(Z, -1. / 3.);
    c.Z23 = std::pow(Z, 2. / 3.);
    c.dn = 1.54 * std::pow(A, 0.27);
    c.lnA = std::log(A);
    c.shadow_low = std::exp(-0.1 * c.lnA);
    const double m = mass * 1E+03;
    const double mu_qc = m / (SSR_MMU * G.e1 / c.dn);
    const double rho = std::sqrt(1. + 4. * mu_qc * mu_qc);
    const double log_rho = std::log((rho + 1.) / (rho - 1.));
    c.b_delta1 = std::log(mu_qc) + 0.5 * rho * log_rho;
    c.b_delta2 = std::log(mu_qc) + 0.25 * (3. * rho - rho * rho * rho) * log_rho + 2. * mu_qc * mu_qc;
    return c;
}

inline void make_grid(double cutoff, Grid& g, EnvelopeGrid& eg) {
#pragma clang fp contract(off)
    const int n = n_table(cutoff);
    g.n = n;
    g.cutoff = cutoff;
    const int p = N_REVERSE;
    const int m = n - p;
    double xrev;
    if (m > 0) {
        xrev = X_REVERSE;
        const double x0 = std::log(cutoff);
        const double dx = std::log(xrev / cutoff) / (m - 1);
        for (int i = 0; i < m; i++) g.x[i] = x0 + i * dx;
        eg.x0 = x0;
        eg.dx = dx;
    } else {
        xrev = cutoff;
    }
    const double dx = std::log((MAX_FRACTION - xrev) / DXMIN) / ((m > 0) ? p : p - 1);
    for (int i = 0; i < p; i++) g.x[n - 1 - i] = std::log(MAX_FRACTION - DXMIN * std::exp(i * dx));
    eg.m = m;
    for (int i = 0; i < p; i++) eg.tail[i] = float(g.x[m + i]);
}

}  // namespace pumas
}  // namespace noa_hip

using namespace noa_hip;

extern "C" {

int noa_pumas_n_table_dcs(double cutoff) {
    if (!(cutoff > 0.0 && cutoff < 1.0)) return fail(NOA_DCS_EINVAL, "cutoff must be in (0, 1) (got %g)", cutoff);
    const int n = pumas::n_table(cutoff);
    if (n > pumas::MAX_X) return fail(NOA_DCS_ERANGE, "cutoff %g needs %d grid nodes, more than %d", cutoff, n,
                                      pumas::MAX_X);
    return n;
}

int noa_pumas_dcs_f64(int32_t process, double Z, double A, double mass, const double* K, const double* q, int64_t n,
                      double* out, hipStream_t stream) {
    if (process < 0 || process > 2) return fail(NOA_DCS_EINVAL, "process must be 0, 1 or 2 (got %d)", process);
    if (!(Z >= 1.0) || !(A > 0.0) || !(mass > 0.0)) return fail(NOA_DCS_EINVAL, "Z >= 1, A > 0 and mass > 0 required");
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (n == 0) return ok();
    if (!K || !q || !out) return fail(NOA_DCS_EINVAL, "K, q and out must be non-NULL");
    const pumas::Globals G = pumas::make_globals();
    const pumas::ElementConsts c = pumas::make_element(Z, A, mass, G);
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(pumas::pumas_dcs_kernel, dim3(unsigned(blocks < 65536 ? blocks : 65536)), dim3(256), 0, stream,
                       int(process), c, G, mass, K, q, n, out);
    if (int rc = check_hip(hipGetLastError(), "pumas_dcs_kernel")) return rc;
    return ok();
}

int noa_pumas_dcs_table(const double* Z, const double* A, int32_t n_elements, double mass, double cutoff,
                        const double* K, int32_t n_K, float* table, float* x, float* envelope, double* table_f64,
                        const double* csn, hipStream_t stream) {
    const int n = noa_pumas_n_table_dcs(cutoff);
    if (n < 0) return n;
    if (n_elements < 0 || n_K < 0) return fail(NOA_DCS_EINVAL, "n_elements and n_K must be >= 0");
    if (!(mass > 0.0)) return fail(NOA_DCS_EINVAL, "mass must be > 0 (got %g)", mass);
    if (int64_t(3) * n_elements * n_K == 0) return ok();
    if (int64_t(3) * 16 * n_K > int64_t(0x7fffffff)) return fail(NOA_DCS_ERANGE, "n_K too large (%d)", n_K);
    if (!Z || !A || !K || !table) return fail(NOA_DCS_EINVAL, "Z, A, K and table must be non-NULL");
    for (int e = 0; e < n_elements; e++)
        if (!(Z[e] >= 1.0) || !(A[e] > 0.0))
            return fail(NOA_DCS_EINVAL, "element %d: Z >= 1 and A > 0 required (got %g, %g)", e, Z[e], A[e]);
    pumas::Grid g;
    pumas::EnvelopeGrid eg{};
    pumas::make_grid(cutoff, g, eg);
    const pumas::Globals G = pumas::make_globals();
    // launches of equal numbers of elements
    const auto per_launch = [&](int room) {
        const int launches = (n_elements + room - 1) / room;
        return (n_elements + launches - 1) / launches;
    };
    for (int e0 = 0, per = per_launch(pumas::MAX_EL); e0 < n_elements; e0 += per) {
        const int n_blk = std::min(n_elements - e0, per);
        pumas::ElementBlock blk{};
        for (int j = 0; j < n_blk; j++) blk.e[j] = pumas::make_element(Z[e0 + j], A[e0 + j], mass, G);
        const int room = pumas::TABLE_WG / g.n;
        const int64_t workgroups = int64_t(3) * n_blk * ((n_K + room - 1) / room);
        const int rc = launch_slices(workgroups, pumas::TABLE_WG, [&](int64_t start, uint32_t count) {
            hipLaunchKernelGGL(pumas::pumas_table_kernel, dim3(count), dim3(pumas::TABLE_WG), 0, stream, g, blk, G,
                               start, e0, n_blk, n_elements, mass, K, n_K, table, table_f64, e0 == 0 ? x : nullptr,
                               envelope, csn);
            return check_hip(hipGetLastError(), "pumas_table_kernel");
        });
        if (rc) return rc;
    }
    if (envelope) {
        hipLaunchKernelGGL(pumas::pumas_alpha_fill_kernel, dim3(unsigned(3 * n_elements)), dim3(64), 0, stream,
                           envelope, n_K);
        if (int rc = check_hip(hipGetLastError(), "pumas_alpha_fill_kernel")) return rc;
        // the envelope maxima, over the finished rows and exponents
        pumas::EnvelopeArgs args{};
        args.g = eg;
        args.G = G;
        args.n_x = g.n;
        args.n_el = n_elements;
        args.mass = mass;
        args.cutoff = cutoff;
        args.Ks = K;
        args.table = table;
        args.csn = csn;
        args.env = envelope;
        args.n_K = n_K;
        for (int per = per_launch(pumas::MAX_ENV_EL); args.e0 < n_elements; args.e0 += per) {
            args.n_blk = std::min(n_elements - args.e0, per);
            for (int j = 0; j < args.n_blk; j++)
                args.blk.e[j] = pumas::make_element(Z[args.e0 + j], A[args.e0 + j], mass, G);
            const int64_t rows = int64_t(3) * args.n_blk * n_K;
            // three waves per SIMD (40 registers spilled) where the rows are many;
            // below, the longest rows decide. Measured (us, two / three waves,
            // 146 energies): 7 elements 548 / 564, 16 575 / 595, 20 632 / 605,
            // 48 1171 / 947
            const auto kernel = rows > 8000 ? &pumas::pumas_envelope_kernel<3> : &pumas::pumas_envelope_kernel<2>;
            const int rc = launch_slices(rows, 64, [&](int64_t start, uint32_t count) {
                args.start = start;
                hipLaunchKernelGGL(kernel, dim3(count), dim3(64), size_t(pumas::ENVELOPE_LDS) * g.n * sizeof(float),
                                   stream, args);
                return check_hip(hipGetLastError(), "pumas_envelope_kernel");
            });
            if (rc) return rc;
        }
    }
    return ok();
}

}  // extern "C"
