// hermite.hip -- batched FP64 4th-order Hermite with block time steps (hard part),
// Kepler drift and Sun-only Hermite for isolated particles.
//
// One workgroup integrates one cluster over local time [0, dt_tree] exactly as
// timeIntegrate_multi does (src/hermite.h:224-479): a block step picks the minimum
// time+dt, predicts every particle, checks collisions (perfect merging), corrects
// the active particles with two P(EC) iterations and updates their block steps.
// The active particles of one block step are independent (each reads only the
// predicted positions of the others), so they are corrected in parallel.  Clusters of 2 to
// 4 bodies hold their state in registers (integrate_pair, integrate_terms), those of up to HERMITE_LDS in
// LDS (hermite_lds.hpp), larger ones in global memory.
// The kernels are persistent: workgroups pull clusters (costliest first: estimated block
// steps times size) from an atomic queue until it is empty.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "hermite.hpp"

namespace gplum {

#define SECONDORDER 5.e-1
#define THIRDORDER 1.6666666666666667e-1
#define ALPHA_POS 1.1666666666666667e-3  // ALPHA = 7/6000 of the corrector's position term, src/particle.h:339 (kept as written)
#define ONE_TWELFTH 8.3333333333333333e-2
#define ONE_SIXTIETH 1.6666666666666667e-2

struct HP {                                  // physics constants for the kernels
    double m_sun, eps2, eps2_sun, dt_tree, dt_min, eta, eta_0, eta_sun, eta_sun0, alpha2;
    Cutoff cut;
    int collision;
    int terms_max;     // clusters of 2 .. terms_max (<= 4) bodies run integrate_pair, integrate_terms
};

__device__ inline double dmin(double a, double b) { return (b < a) ? b : a; }

// collisionDetermination looks for R = |dx| / (f_i R_i + f_j R_j) < 1.  Pairs with
// |dx|^2 >= (1 + 1e-10) (f_i R_i + f_j R_j)^2 have R >= 1 even after the rounding of
// sqrt and the division, so they are skipped before computing R; the minimum and its
// pair are unchanged.
constexpr double COL_FILTER = 1.0 + 1e-10;

// ------------------------------------------- square roots and reciprocals together
//
// A force term needs sqrt(s) and 1 / sqrt(s), or 1 / s and its square root, each correctly
// rounded.  One hardware estimate of 1 / sqrt(s) serves both: a Goldschmidt step gives g ~
// sqrt(s) and h ~ 1 / (2 sqrt(s)) to about 2^-45, and two residual corrections (the residual
// exact by FMA, the second one the rounding step) give the correctly rounded root, and two
// Newton steps the correctly rounded reciprocal (Markstein, IBM J. Res. Dev. 34, 1990).  The
// library's sqrt takes the same corrections after scaling, its division starts over from the
// estimate of 1 / b; in range there is nothing to scale, and a wave with a value out of range
// calls the library.  gplum_hermite_path_selfcheck compares the results with sqrt and 1 / x bit for
// bit.  sqrt and division in sequence took 92 + 70 cycles of latency (dependent FP64
// operations 7 cycles, the estimate 18); here 18 + 14 operations.

// s in [2^-400, 2^401): roots and reciprocals are normal and nothing is scaled
__device__ inline bool root_range(double s) {
    const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(s) >> 32);
    return hi - (623u << 20) < (801u << 20);
}
// rcp_fix rounds correctly unless b's mantissa is all ones: a low word of ones (one value in
// 2^32) goes to the library too
__device__ inline bool rcp_exception(double b) { return (int)__double_as_longlong(b) == -1; }
__device__ inline void root_seed(double s, double &g, double &h) {
    const double y = __builtin_amdgcn_rsq(s);
    g = s * y;
    h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(g, r, g);
}
// sqrt(x) from g ~ sqrt(x) and h ~ 1 / (2 sqrt(x))
__device__ inline double root_fix(double x, double g, double h) {
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
// 1 / b from y ~ 1 / b
__device__ inline double rcp_fix(double b, double y) {
    y = __builtin_fma(__builtin_fma(-b, y, 1.), y, y);
    return __builtin_fma(__builtin_fma(-b, y, 1.), y, y);
}
// r = sqrt(s) and rinv = 1 / r (need: the values are used; otherwise anything may come back)
__device__ inline void root_and_inverse(double s, bool need, double &r, double &rinv) {
    double g, h;
    root_seed(s, g, h);
    r = root_fix(s, g, h);
    rinv = rcp_fix(r, 2. * h);
    if (__ballot(need && (!root_range(s) || rcp_exception(r)))) {
        r = sqrt(s);
        rinv = 1. / r;
    }
}
// sinv = 1 / s and rinv = sqrt(sinv)
__device__ inline void inverse_and_root(double s, double &sinv, double &rinv) {
    double g, h;
    root_seed(s, g, h);
    const double y = 2. * h;
    sinv = rcp_fix(s, y * y);
    rinv = root_fix(sinv, y, 0.5 * g);
    if (__ballot(!root_range(s) || rcp_exception(s))) {
        sinv = 1. / s;
        rinv = sqrt(sinv);
    }
}

// ---------------------------------------------------------- Sun gravity

__device__ inline void star_acc_jerk(const HP &P, const double x[3], const double v[3],
                                     double acc[3], double jerk[3], double *phi) {
    const double dr[3] = {-x[0], -x[1], -x[2]};
    const double dv[3] = {-v[0], -v[1], -v[2]};
    double r2inv, rinv;
    inverse_and_root(dot3(dr[0], dr[1], dr[2], dr[0], dr[1], dr[2]) + P.eps2_sun, r2inv, rinv);
    const double r3inv = rinv * r2inv;
    const double mj = P.m_sun * r3inv;
    const double alpha = dot3(dr[0], dr[1], dr[2], dv[0], dv[1], dv[2]) * r2inv;
    if (phi) *phi = -P.m_sun * rinv;
    for (int k = 0; k < 3; k++) {
        acc[k] = mj * dr[k];
        jerk[k] = mj * (dv[k] - 3. * alpha * dr[k]);
    }
}

// -------------------------------------------------------------- time steps

__device__ inline double calc_dt2(double eta, double alpha2, double acc0, const double a[3],
                                  const double j[3]) {
    const double Acc2 = dot3(a[0], a[1], a[2], a[0], a[1], a[2]) + alpha2 * acc0 * acc0;
    const double Jerk2 = dot3(j[0], j[1], j[2], j[0], j[1], j[2]);
    return (Jerk2 > 0.) ? eta * sqrt(Acc2 / Jerk2) : DBL_MAX;
}
__device__ inline double calc_dt4(double eta, double alpha2, double acc0, const double a[3],
                                  const double j[3], const double s[3], const double c[3]) {
    const double Acc = sqrt(dot3(a[0], a[1], a[2], a[0], a[1], a[2]) + alpha2 * acc0 * acc0);
    const double Jerk2 = dot3(j[0], j[1], j[2], j[0], j[1], j[2]);
    const double Jerk = sqrt(Jerk2);
    const double Snap2 = dot3(s[0], s[1], s[2], s[0], s[1], s[2]);
    const double Snap = sqrt(Snap2);
    const double Crac = sqrt(dot3(c[0], c[1], c[2], c[0], c[1], c[2]));
    return (Jerk > 0.) ? eta * sqrt((Acc * Snap + Jerk2) / (Jerk * Crac + Snap2)) : DBL_MAX;
}

// FPGrav::calcDeltatInitial, src/particle.h:886-914.
__device__ inline double dt_initial(const HP &P, double time, double dt, double acc0,
                                    const double acc_d[3], const double jerk_d[3],
                                    const double acc_s[3], const double jerk_s[3]) {
    double dt_next = 0.5 * P.dt_tree;
    const double dt_1 = dmin(calc_dt2(P.eta_0, P.alpha2, acc0, acc_d, jerk_d),
                             calc_dt2(P.eta_sun0, P.alpha2, 0., acc_s, jerk_s));
    double rem = fmod_block(time, dt_next);
    for (int it = 0; rem != 0.0 && it < HALVE_CAP; it++) { dt_next *= 0.5; rem = fmod_block(time, dt_next); }
    if (rem != 0.0) return P.dt_min;
    if (dt > 0.)
        for (int it = 0; 2. * dt < dt_next && it < HALVE_CAP; it++) dt_next *= 0.5;
    for (int it = 0; dt_1 < dt_next && it < HALVE_CAP; it++) dt_next *= 0.5;
    if (dt_next < 2. * P.dt_min) dt_next = P.dt_min;
    return dt_next;
}

// calc_dt4 with the hardware square root and reciprocal (v_sqrt_f64, v_rcp_f64, not
// correctly rounded; Acc * Snap as sqrt(Acc2 * Snap2), Jerk * Crac likewise): within a
// few 1e-7 of calc_dt4 relative, DBL_MAX exactly where calc_dt4 gives it (Jerk > 0 iff
// Jerk2 > 0).  A product that underflows (0 from non-zero factors, or subnormal) gives
// NaN and one that overflows gives inf or NaN; dt_block sends either to calc_dt4.
__device__ inline double calc_dt4_fast(double eta, double alpha2, double acc0, const double a[3],
                                       const double j[3], const double s[3], const double c[3]) {
    const double Acc2 = dot3(a[0], a[1], a[2], a[0], a[1], a[2]) + alpha2 * acc0 * acc0;
    const double Jerk2 = dot3(j[0], j[1], j[2], j[0], j[1], j[2]);
    const double Snap2 = dot3(s[0], s[1], s[2], s[0], s[1], s[2]);
    const double Crac2 = dot3(c[0], c[1], c[2], c[0], c[1], c[2]);
    // selects, not branches: the Sun and planet criteria of dt_block stay one basic block
    const double as2 = Acc2 * Snap2, jc2 = Jerk2 * Crac2;
    const bool ok = (as2 >= DBL_MIN || (Acc2 == 0. || Snap2 == 0.)) && (jc2 >= DBL_MIN || Crac2 == 0.);
    const double num = __builtin_amdgcn_sqrt(as2) + Jerk2;
    const double den = __builtin_amdgcn_sqrt(jc2) + Snap2;
    const double q = ok ? eta * __builtin_amdgcn_sqrt(num * __builtin_amdgcn_rcp(den)) : __builtin_nan("");
    return (Jerk2 > 0.) ? q : DBL_MAX;
}

// True when t is farther than 2^-10 relative from every d * 2^k (k integer), for
// t > 2^-1000 and finite: then t and any value within 2^-11 of it relative lie on the
// same side of each of those grid points.  t = m_t 2^e_t, d = m_d 2^e_d with mantissas
// in [0.5, 1): the grid points nearest t are at m_t / m_d in {1/2, 1, 2}.
__device__ inline bool clear_of_grid(double t, double d) {
    int et = 0, ed = 0;
    const double r = frexp(t, &et) * __builtin_amdgcn_rcp(frexp(d, &ed));
    const double tol = 0x1p-10;
    return (t > 0x1p-1000 && t < DBL_MAX) && r > 0.5 * (1. + tol) && (r < 1. - tol || r > 1. + tol) &&
           r < 2. * (1. - tol);
}

// FPHard::calcDeltat, src/particle.h:1276-1314.  dt_1 enters the result only through
// dt_1 < dt_next for dt_next = D, D/2, D/4, ... (D the step left by the fmod loop,
// halvings exact above 2^-1000), so a dt_1 from calc_dt4_fast that is clear of that
// grid decides every comparison as the correctly rounded dt_1 does; near the grid, or
// when either fast criterion is NaN or infinite (under- or overflow of its products,
// which the minimum would otherwise drop), calc_dt4 itself is evaluated.  Same result,
// bit for bit.
// FAST = false: calc_dt4 always (the self-check's reference).
template <bool FAST = true>
__device__ inline double dt_block(const HP &P, double time, double dt, double acc0,
                                  const double acc_d[3], const double jerk_d[3], const double a2_d[3],
                                  const double a3_d[3], const double acc_s[3], const double jerk_s[3],
                                  const double a2_s[3], const double a3_s[3], int *fell_back = nullptr) {
    double dt_next = dmin(2. * dt, 0.5 * P.dt_tree);
    double rem = fmod_block(time, dt_next);
    for (int it = 0; rem != 0.0 && it < HALVE_CAP; it++) { dt_next *= 0.5; rem = fmod_block(time, dt_next); }
    if (rem != 0.0) return P.dt_min;
    double dt_1 = 0.;
    bool exact = !FAST;
    if (FAST) {
        const double f_planet = calc_dt4_fast(P.eta, P.alpha2, acc0, acc_d, jerk_d, a2_d, a3_d);
        const double f_sun = calc_dt4_fast(P.eta_sun, P.alpha2, 0., acc_s, jerk_s, a2_s, a3_s);
        dt_1 = dmin(f_planet, f_sun);
        // DBL_MAX is a valid value (no jerk); NaN and inf are not
        exact = !(f_planet <= DBL_MAX && f_sun <= DBL_MAX) || !clear_of_grid(dt_1, dt_next);
        if (fell_back) *fell_back = exact ? 1 : 0;
    }
    if (exact)
        dt_1 = dmin(calc_dt4(P.eta, P.alpha2, acc0, acc_d, jerk_d, a2_d, a3_d),
                    calc_dt4(P.eta_sun, P.alpha2, 0., acc_s, jerk_s, a2_s, a3_s));
    for (int it = 0; dt_1 < dt_next && 0.5 * dt < dt_next && it < HALVE_CAP; it++) dt_next *= 0.5;
    if (dt_next < 2. * P.dt_min) dt_next = P.dt_min;
    return dt_next;
}

// Whether d is a power of two (normal, 2^-999 to 2^999): then 1/d, and products with it, are
// exact.  Every block step is one (dt_tree halved some times).
__host__ __device__ inline bool is_pow2(double d) {
    unsigned long long b;
    __builtin_memcpy(&b, &d, sizeof b);
    const unsigned hi = (unsigned)(b >> 32);
    return ((unsigned)b | (hi & 0xFFFFFu)) == 0u && hi - (24u << 20) <= (1998u << 20);
}
__device__ inline double pow2_inverse(double d) {
    return __longlong_as_double(0x7FE0000000000000ll - __double_as_longlong(d));
}
// recip_block without its frexp and ldexp
__device__ inline double recip_step(double d) {
    if (is_pow2(d)) return pow2_inverse(d);
    return recip_block(d);
}

// The first part of dt_block: dt_max halved until it divides time (cap: it never did).
__device__ inline double dt_candidate(double time, double dt_max, bool &cap) {
    double d = dt_max;
    if (is_pow2(d) && time >= 0.) {
        double q = time * pow2_inverse(d);          // exact, so q is whole iff d divides time
        int it = 0;
        for (; q != floor(q) && it < HALVE_CAP; it++) { q *= 2.; d *= 0.5; }
        cap = it == HALVE_CAP;
    } else {
        double rem = fmod_block(time, d);
        for (int it = 0; rem != 0.0 && it < HALVE_CAP; it++) { d *= 0.5; rem = fmod_block(time, d); }
        cap = rem != 0.0;
    }
    return d;
}
// Its last part: dt_0 halved while it exceeds both dt_1 and dt / 2 (twice at most when dt_0
// <= 2 dt).
__device__ inline double dt_reduce(double dt_0, double dt_1, double dt) {
    double d = dt_0;
    if (dt_0 <= 2. * dt) {
        for (int it = 0; it < 2; it++) d = (dt_1 < d && 0.5 * dt < d) ? 0.5 * d : d;
    } else {
        for (int it = 0; dt_1 < d && 0.5 * dt < d && it < HALVE_CAP; it++) d *= 0.5;
    }
    return d;
}
// clear_of_grid for a power of two d from t's mantissa bits (a slightly narrower range)
__device__ inline bool clear_of_steps(double t, double d) {
    if (!is_pow2(d)) return clear_of_grid(t, d);
    const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(t) >> 32);
    return (hi & 0xFFFFFu) - 1025u < 0x100000u - 2049u - 1025u && hi - (24u << 20) <= (1998u << 20);
}

// ------------------------------------------------------------- hard pair

// K(x) and dK/dr of cutfunc.h with selects (the polynomial evaluated everywhere).
__device__ inline double cutoff_K_sel(const Cutoff &c, double rij, double r_out_inv) {
    const double x = (c.gamma - rij * r_out_inv) * c.g_1_inv;
    const double x2 = x * x;
    const double p = (((-20. * x + 70.) * x - 84.) * x + 35.) * x2 * x2;
    return (x < 0.) ? 0. : ((x >= 1.) ? 1. : p);
}
__device__ inline double cutoff_dKdt_sel(const Cutoff &c, double rij, double r_out_inv, double alpha) {
    const double x = (c.gamma - rij * r_out_inv) * c.g_1_inv;
    const double x_1 = x - 1.;
    const double d = 140. * x * x * x * x_1 * x_1 * x_1 * r_out_inv * c.g_1_inv;
    const double dKdr = (x < 0. || x >= 1.) ? 0. : d;
    return alpha * rij * dKdr;
}

// gravity_hard.h:219-255: the summands of acc_d, jerk_d (and phi_d) of i from j,
// returned separately so that several j can be evaluated side by side and added in
// ascending j afterwards (the sums stay those of a sequential loop).  need: the summands are
// used (the pair of a particle with itself, at distance 0, is evaluated and dropped).
__device__ inline void pair_term(const HP &P, const double xi[3], const double vi[3], double rinv_i,
                                 double xj0, double xj1, double xj2, double vj0, double vj1, double vj2,
                                 double mj, double rinv_j, double ta[3], double tj[3], double *tphi,
                                 bool need = true) {
    const double dr[3] = {xj0 - xi[0], xj1 - xi[1], xj2 - xi[2]};
    double dr2 = dot3(dr[0], dr[1], dr[2], dr[0], dr[1], dr[2]);
    dr2 += P.eps2;
    const double dv[3] = {vj0 - vi[0], vj1 - vi[1], vj2 - vi[2]};
    double rij, rinv;
    root_and_inverse(dr2, need, rij, rinv);
    const double r2inv = rinv * rinv;
    const double r3inv = r2inv * rinv;
    const double r_out_inv = dmin(rinv_i, rinv_j);
    const double mj_rij3 = mj * r3inv;
    const double alpha = dot3(dr[0], dr[1], dr[2], dv[0], dv[1], dv[2]) * r2inv;
    const double _K = 1. - cutoff_K_sel(P.cut, rij, r_out_inv);
    const double dKdt = cutoff_dKdt_sel(P.cut, rij, r_out_inv, alpha);
    const double alpha_c = alpha * _K;
    if (tphi) {
        const double _W = 1. - cutoff_W(P.cut, rij, r_out_inv);
        *tphi = mj * rinv * _W;
    }
    const double c2 = 3. * alpha_c + dKdt;
    for (int k = 0; k < 3; k++) {
        ta[k] = mj_rij3 * _K * dr[k];
        tj[k] = mj_rij3 * (_K * dv[k] - c2 * dr[k]);
    }
}

// ---------------------------------------------------------- cluster state

struct HardView {          // SoA arrays of the gathered cluster particles
    double *pos, *vel, *acc_s, *jerk_s, *acc_d, *jerk_d, *xp, *vp, *a0_s, *j0_s, *a0_d, *j0_d;
    double *a2_s, *a3_s, *a2_d, *a3_d;                       // 3 per particle
    double *mass, *rinv, *time, *dt, *acc0, *r_planet, *f, *phi_d, *phi_s;
    int64_t *id;
    int32_t *flags, *twin_of, *act;     // act: active in the current block step
    // collision records (COLREC doubles each, see perfect_merge), when the caller keeps a
    // collision log: crec null otherwise
    double *crec;
    unsigned *ccount;
    unsigned ccap;
    int base;              // index of the arrays' first element among all clusters' particles
};

// The clusters of one launch: offsets, processing order (or null), queue and outcomes.
struct ClusterArgs {
    const int32_t *off, *order;
    int ncl, persistent;
    int *next;
    double *edisp;
    int *ncol;
    long long *nblock, *npair;
};

__device__ inline void ld3(const double *a, int i, double v[3]) {
    v[0] = a[3 * i]; v[1] = a[3 * i + 1]; v[2] = a[3 * i + 2];
}
__device__ inline void st3(double *a, int i, const double v[3]) {
    a[3 * i] = v[0]; a[3 * i + 1] = v[1]; a[3 * i + 2] = v[2];
}

// j-data accessor: LDS when the cluster fits, else global memory.
struct JData {
    const double *x, *v, *m, *ri;
    const int64_t *id;
};

// pairs evaluated side by side per lane (independent dependency chains; the one wave
// of a small cluster has no other wave to hide FP64 latency behind)
constexpr int HARD_ILP = 4;

__device__ inline void pair_term_j(const HP &P, const JData &J, int j, const double xi[3], const double vi[3],
                                   double rinv_i, double ta[3], double tj[3], double *tphi, bool need = true) {
    pair_term(P, xi, vi, rinv_i, J.x[3 * j], J.x[3 * j + 1], J.x[3 * j + 2], J.v[3 * j], J.v[3 * j + 1],
              J.v[3 * j + 2], J.m[j], J.ri[j], ta, tj, tphi, need);
}

// Sum over j = j0, j0 + s, j0 + 2s, ... < n (j != i by id) in ascending j, ILP pairs
// evaluated at a time.  The self pair is evaluated too (its summands may be NaN) and
// not added.
template <int ILP = HARD_ILP>
__device__ inline void pair_sum_strided(const HP &P, const JData &J, int j0, int s, int n, int64_t idi,
                                        const double xi[3], const double vi[3], double rinv_i, double acc[3],
                                        double jerk[3], double *phi) {
    int j = j0;
    for (; j + (ILP - 1) * s < n; j += ILP * s) {
        double ta[ILP][3], tj[ILP][3], tp[ILP];
        bool use[ILP];
#pragma unroll
        for (int u = 0; u < ILP; u++) {
            use[u] = J.id[j + u * s] != idi;
            pair_term_j(P, J, j + u * s, xi, vi, rinv_i, ta[u], tj[u], phi ? &tp[u] : nullptr, use[u]);
        }
#pragma unroll
        for (int u = 0; u < ILP; u++) {
            if (!use[u]) continue;
            for (int k = 0; k < 3; k++) { acc[k] += ta[u][k]; jerk[k] += tj[u][k]; }
            if (phi) *phi -= tp[u];
        }
    }
    for (; j < n; j += s) {
        if (J.id[j] == idi) continue;
        double ta[3], tj[3], tp;
        pair_term_j(P, J, j, xi, vi, rinv_i, ta, tj, phi ? &tp : nullptr);
        for (int k = 0; k < 3; k++) { acc[k] += ta[k]; jerk[k] += tj[k]; }
        if (phi) *phi -= tp;
    }
}

__device__ inline void gravity_loop(const HP &P, const JData &J, int n, int64_t idi,
                                    const double xi[3], const double vi[3], double rinv_i,
                                    double acc[3], double jerk[3], double *phi) {
    acc[0] = acc[1] = acc[2] = 0.;
    jerk[0] = jerk[1] = jerk[2] = 0.;
    pair_sum_strided(P, J, 0, 1, n, idi, xi, vi, rinv_i, acc, jerk, phi);
}

// gravity_loop with one lane per particle, for clusters whose ids are known to be distinct: lane
// i's partners are j = k + (k >= i) for k = 0 .. n-2, ascending j as in gravity_loop, so every
// lane runs the same n-1 iterations (the loop over all j with a self test would run n iterations
// with one lane masked off in each).
__device__ inline void gravity_loop_lane(const HP &P, const JData &J, int n, int i, const double xi[3], const double vi[3],
                                         double rinv_i, double acc[3], double jerk[3], double *phi) {
    acc[0] = acc[1] = acc[2] = 0.;
    jerk[0] = jerk[1] = jerk[2] = 0.;
    const int m = n - 1;
    int k = 0;
    for (; k + HARD_ILP <= m; k += HARD_ILP) {
        double ta[HARD_ILP][3], tj[HARD_ILP][3], tp[HARD_ILP];
#pragma unroll
        for (int u = 0; u < HARD_ILP; u++)
            pair_term_j(P, J, k + u + ((k + u) >= i ? 1 : 0), xi, vi, rinv_i, ta[u], tj[u], phi ? &tp[u] : nullptr);
#pragma unroll
        for (int u = 0; u < HARD_ILP; u++) {
            for (int d = 0; d < 3; d++) {
                acc[d] += ta[u][d];
                jerk[d] += tj[u][d];
            }
            if (phi) *phi -= tp[u];
        }
    }
    for (; k < m; k++) {
        double ta[3], tj[3], tp;
        pair_term_j(P, J, k + (k >= i ? 1 : 0), xi, vi, rinv_i, ta, tj, phi ? &tp : nullptr);
        for (int d = 0; d < 3; d++) {
            acc[d] += ta[d];
            jerk[d] += tj[d];
        }
        if (phi) *phi -= tp;
    }
}

// calcGravity (full, with phi_d and Sun phi), gravity_hard.h:203-256, current pos/vel.
__device__ void gravity_full(const HP &P, HardView &H, int b, int n, int i) {
    double x[3], v[3], as[3], js[3], ad[3], jd[3], phs, phd = 0.;
    ld3(H.pos, b + i, x);
    ld3(H.vel, b + i, v);
    star_acc_jerk(P, x, v, as, js, &phs);
    const JData Jc{H.pos + 3 * b, H.vel + 3 * b, H.mass + b, H.rinv + b, H.id + b};
    gravity_loop(P, Jc, n, H.id[b + i], x, v, H.rinv[b + i], ad, jd, &phd);
    st3(H.acc_s, b + i, as);
    st3(H.jerk_s, b + i, js);
    st3(H.acc_d, b + i, ad);
    st3(H.jerk_d, b + i, jd);
    H.phi_s[b + i] = phs;
    H.phi_d[b + i] = phd;
}

// FPHard::predict, src/particle.h:1183-1207.
__device__ inline void predict(HardView &H, int g, double Dt) {
    for (int k = 0; k < 3; k++) {
        const double pos = H.pos[3 * g + k], vel = H.vel[3 * g + k];
        const double as = H.acc_s[3 * g + k], ad = H.acc_d[3 * g + k];
        const double js = H.jerk_s[3 * g + k], jd = H.jerk_d[3 * g + k];
        H.a0_s[3 * g + k] = as;
        H.j0_s[3 * g + k] = js;
        H.j0_d[3 * g + k] = jd;
        H.a0_d[3 * g + k] = ad;
        const double acc_sd = as + ad;
        const double jerk_sd = js + jd;
        H.xp[3 * g + k] = pos + Dt * (vel + Dt * (SECONDORDER * acc_sd + THIRDORDER * Dt * jerk_sd));
        H.vp[3 * g + k] = vel + Dt * (acc_sd + Dt * SECONDORDER * jerk_sd);
    }
}

__device__ inline void correct_regs(double Dt, const double xp[3], const double vp[3], const double as[3],
                                    const double a0s[3], const double j0s[3], const double js[3], const double ad[3],
                                    const double a0d[3], const double j0d[3], const double jd[3], double pos[3],
                                    double vel[3], double a2s[3], double a3s[3], double a2d[3], double a3d[3]) {
    const double Dt2 = Dt * Dt;
    const double Dt_inv = recip_block(Dt);
    const double Dt_inv2 = Dt_inv * Dt_inv;
    const double Dt_inv3 = Dt_inv2 * Dt_inv;
    for (int k = 0; k < 3; k++) {
        const double Am_s = as[k] - a0s[k];
        const double J0_s = Dt * j0s[k];
        const double J1_s = Dt * js[k];
        const double A2_s = 3. * Am_s - (J1_s + 2. * J0_s);
        const double A3_s = -2. * Am_s + (J1_s + J0_s);
        a2s[k] = 2. * Dt_inv2 * (A2_s + 3. * A3_s);
        a3s[k] = 6. * Dt_inv3 * A3_s;
        const double Am_d = ad[k] - a0d[k];
        const double J0_d = j0d[k] * Dt;
        const double J1_d = jd[k] * Dt;
        const double A2_d = 3. * Am_d - (J1_d + 2. * J0_d);
        const double A3_d = -2. * Am_d + (J1_d + J0_d);
        a2d[k] = 2. * (A2_d + 3. * A3_d) * Dt_inv2;
        a3d[k] = 6. * A3_d * Dt_inv3;
        const double A2_sd = A2_s + A2_d;
        const double A3_sd = A3_s + A3_d;
        pos[k] = xp[k] + ONE_SIXTIETH * Dt2 * (5. * A2_sd + 3. * ALPHA_POS * A3_sd);
        vel[k] = vp[k] + ONE_TWELFTH * Dt * (4. * A2_sd + 3. * A3_sd);
    }
}

// Hard force on one particle with all 64 lanes of the (one-wave) workgroup: lane l
// sums the pairs j = l, l+64, ... in ascending j, then a butterfly over the lanes adds
// the 64 partial sums (every lane ends with the same total).  This fixed order is the
// hard-force summation order of clusters above HARD_SEQ_MAX particles (the oracle sums
// the same way); smaller clusters sum sequentially in j.
// Lane permutations within rows of 16 lanes (DPP): quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror, row_mirror.  Applied in this order with a min, they
// leave every lane of a row holding the row's minimum.
constexpr int DPP_QUAD_1032 = 0xB1, DPP_QUAD_2301 = 0x4E, DPP_ROW_HALF_MIRROR = 0x141, DPP_ROW_MIRROR = 0x140;
// quad_perm [3,2,1,0] and row_ror:8 (rotate a row of 16 lanes by 8: lane ^ 8)
constexpr int DPP_QUAD_3210 = 0x1B, DPP_ROW_ROR8 = 0x128;

template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ inline double readlane_f64(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ inline void coop_pair_sum(const HP &P, const JData &J, int n, int64_t idi, const double xi[3],
                                     const double vi[3], double rinv_i, double acc[3], double jerk[3]) {
    double a[3] = {0., 0., 0.}, jk[3] = {0., 0., 0.};
    // two pairs at a time: the callers hold much state per lane
    pair_sum_strided<2>(P, J, (int)(threadIdx.x & 63), 64, n, idi, xi, vi, rinv_i, a, jk, nullptr);
    // butterfly x += x[lane ^ d] for d = 32, 16, 8, 4, 2, 1 (every lane active): the two
    // levels across rows of 16 lanes by shuffles, the four inside a row by DPP moves
    // (row_ror:8 is lane ^ 8; quad_perm [3,2,1,0] after row_half_mirror is lane ^ 4;
    // quad_perm [2,3,0,1] and [1,0,3,2] are lane ^ 2 and lane ^ 1), which skip the LDS
    // crossbar.  The same partner values in the same order as the shuffle butterfly.
    for (int d = 32; d > 8; d >>= 1)
        for (int k = 0; k < 3; k++) {
            a[k] += __shfl_xor(a[k], d);
            jk[k] += __shfl_xor(jk[k], d);
        }
    for (int k = 0; k < 3; k++) { a[k] += dpp_f64<DPP_ROW_ROR8>(a[k]); jk[k] += dpp_f64<DPP_ROW_ROR8>(jk[k]); }
    for (int k = 0; k < 3; k++) {
        a[k] += dpp_f64<DPP_QUAD_3210>(dpp_f64<DPP_ROW_HALF_MIRROR>(a[k]));
        jk[k] += dpp_f64<DPP_QUAD_3210>(dpp_f64<DPP_ROW_HALF_MIRROR>(jk[k]));
    }
    for (int k = 0; k < 3; k++) { a[k] += dpp_f64<DPP_QUAD_2301>(a[k]); jk[k] += dpp_f64<DPP_QUAD_2301>(jk[k]); }
    for (int k = 0; k < 3; k++) { a[k] += dpp_f64<DPP_QUAD_1032>(a[k]); jk[k] += dpp_f64<DPP_QUAD_1032>(jk[k]); }
    for (int k = 0; k < 3; k++) { acc[k] = a[k]; jerk[k] = jk[k]; }
}

// mergeAccJerk (hermite.h:36-74) for target t: the mass-weighted mean of the target's
// and its twins' acc_d/jerk_d (each computed with its own cut-off radius), in twin
// index order, written to all of them.
__device__ inline void merge_acc_jerk(HardView &H, int b, int n, int t) {
    double acc[3], jerk[3], mass = H.mass[b + t];
    for (int k = 0; k < 3; k++) {
        acc[k] = H.mass[b + t] * H.acc_d[3 * (b + t) + k];
        jerk[k] = H.mass[b + t] * H.jerk_d[3 * (b + t) + k];
    }
    for (int j = 0; j < n; j++) {
        if (H.twin_of[b + j] != t) continue;
        for (int k = 0; k < 3; k++) {
            acc[k] += H.mass[b + j] * H.acc_d[3 * (b + j) + k];
            jerk[k] += H.mass[b + j] * H.jerk_d[3 * (b + j) + k];
        }
        mass += H.mass[b + j];
    }
    const double minv = 1. / mass;
    for (int k = 0; k < 3; k++) { acc[k] *= minv; jerk[k] *= minv; }
    st3(H.acc_d, b + t, acc);
    st3(H.jerk_d, b + t, jerk);
    for (int j = 0; j < n; j++) {
        if (H.twin_of[b + j] != t) continue;
        st3(H.acc_d, b + j, acc);
        st3(H.jerk_d, b + j, jerk);
    }
}

// Perfect merging (collisionA.h:91-103, 155-356, 358-669; hermite.h:413-423), run
// by one thread.  Returns the dissipated energy.
__device__ double perfect_merge(const HP &P, HardView &H, int b, int n, int ic, int jc) {
    const int I = b + ic, T = b + jc;
    double pos_imp[3], pos_tar[3], vel_imp[3], vel_tar[3];
    ld3(H.pos, I, pos_imp); ld3(H.pos, T, pos_tar);
    ld3(H.vel, I, vel_imp); ld3(H.vel, T, vel_tar);
    double mass_imp = H.mass[I], mass_tar = H.mass[T];
    if (H.flags[I] & GPLUM_FLAG_MERGED)
        for (int a = 0; a < n; a++) if (H.twin_of[b + a] == ic) mass_imp += H.mass[b + a];
    if (H.flags[T] & GPLUM_FLAG_MERGED)
        for (int a = 0; a < n; a++) if (H.twin_of[b + a] == jc) mass_tar += H.mass[b + a];
    double vel_g[3], pos_new[3], vel_new[3];
    for (int k = 0; k < 3; k++) {
        vel_g[k] = (mass_imp * vel_imp[k] + mass_tar * vel_tar[k]) / (mass_imp + mass_tar);
        pos_new[k] = (mass_imp * pos_imp[k] + mass_tar * pos_tar[k]) / (mass_imp + mass_tar);
        vel_new[k] = vel_g[k];
    }
    if (H.crec) {
        // Collision0::write2File's record (collisionA.h:122-148; inputPair, setParticle
        // :155-356 with n_frag = 0): the impactor's cluster-local time, ids, masses with
        // their twins, positions and velocities at the collision, and the relative shifts
        // of the centre of mass, |g_new - g| / |g| for position and velocity, where g =
        // pos_g of inputPair (= pos_new here) and g_new = ((m_imp - 0) pos_new + m_tar
        // pos_new) / (m_imp - 0 + m_tar) of setParticle.  Slot COLREC - 1: the cluster's
        // base index, for the log's cluster order.
        const unsigned k = atomicAdd(H.ccount, 1u);
        if (k < H.ccap) {
            double *r = H.crec + (size_t)k * COLREC;
            double dp[3], dv[3];
            const double mt = mass_imp - 0. + mass_tar;
            for (int q = 0; q < 3; q++) {
                dp[q] = ((mass_imp - 0.) * pos_new[q] + mass_tar * pos_new[q]) / mt - pos_new[q];
                dv[q] = ((mass_imp - 0.) * vel_new[q] + mass_tar * vel_new[q]) / mt - vel_g[q];
            }
            r[0] = H.time[I];
            r[1] = (double)H.id[I];
            r[2] = (double)H.id[T];
            r[3] = mass_imp;
            r[4] = mass_tar;
            for (int q = 0; q < 3; q++) {
                r[5 + q] = pos_imp[q]; r[8 + q] = pos_tar[q];
                r[11 + q] = vel_imp[q]; r[14 + q] = vel_tar[q];
            }
            r[17] = sqrt(dot3(dp[0], dp[1], dp[2], dp[0], dp[1], dp[2]) /
                         dot3(pos_new[0], pos_new[1], pos_new[2], pos_new[0], pos_new[1], pos_new[2]));
            r[18] = sqrt(dot3(dv[0], dv[1], dv[2], dv[0], dv[1], dv[2]) /
                         dot3(vel_g[0], vel_g[1], vel_g[2], vel_g[0], vel_g[1], vel_g[2]));
            r[COLREC - 1] = (double)(H.base + b);
        }
    }
    const double mass_rem = mass_imp + mass_tar;
    H.r_planet[I] = 0.;
    H.r_planet[T] *= cbrt_exact_ops(mass_rem / mass_tar);
    const int64_t tar_id = H.id[T];
    H.id[I] = tar_id;
    H.flags[I] |= GPLUM_FLAG_DEAD;
    for (int a = 0; a < n; a++)
        if (H.twin_of[b + a] == ic) { H.id[b + a] = tar_id; H.flags[b + a] |= GPLUM_FLAG_DEAD; }
    H.flags[T] |= GPLUM_FLAG_MERGED;
    for (int a = 0; a < n; a++) {
        if (a == ic || a == jc || H.twin_of[b + a] == ic || H.twin_of[b + a] == jc) {
            st3(H.pos, b + a, pos_new);
            st3(H.vel, b + a, vel_new);
        }
    }
    // calcEnergyDissipation (n_frag = 0)
    double e_kin = 0., s, vr[3];
    for (int k = 0; k < 3; k++) vr[k] = vel_imp[k] - vel_tar[k];
    s = 0.5 * mass_imp * mass_tar / (mass_imp + mass_tar);
    e_kin -= (s * vr[0]) * vr[0] + (s * vr[1]) * vr[1] + (s * vr[2]) * vr[2];
    for (int k = 0; k < 3; k++) vr[k] = vel_new[k] - vel_g[k];
    s = 0.5 * (mass_imp - 0.);
    e_kin += (s * vr[0]) * vr[0] + (s * vr[1]) * vr[1] + (s * vr[2]) * vr[2];
    s = 0.5 * mass_tar;
    e_kin += (s * vr[0]) * vr[0] + (s * vr[1]) * vr[1] + (s * vr[2]) * vr[2];
    double e_int = 0.;
    const double dr[3] = {pos_imp[0] - pos_tar[0], pos_imp[1] - pos_tar[1], pos_imp[2] - pos_tar[2]};
    const double dr2 = dot3(dr[0], dr[1], dr[2], dr[0], dr[1], dr[2]) + P.eps2;
    const double rinv = sqrt(1. / dr2);
    double dphi = H.mass[I] * rinv;
    e_int += H.mass[T] * dphi;
    for (int a = 0; a < n; a++) if (H.twin_of[b + a] == jc) e_int += H.mass[b + a] * dphi;
    for (int i2 = 0; i2 < n; i2++) {
        if (H.twin_of[b + i2] != ic) continue;
        dphi = H.mass[b + i2] * rinv;
        e_int += H.mass[T] * dphi;
        for (int a = 0; a < n; a++) if (H.twin_of[b + a] == jc) e_int += H.mass[b + a] * dphi;
    }
    double e_sun = 0.;
    e_sun += mass_imp / sqrt(dot3(pos_imp[0], pos_imp[1], pos_imp[2], pos_imp[0], pos_imp[1], pos_imp[2]) + P.eps2) +
             mass_tar / sqrt(dot3(pos_tar[0], pos_tar[1], pos_tar[2], pos_tar[0], pos_tar[1], pos_tar[2]) + P.eps2);
    double d2 = dot3(H.pos[3 * T], H.pos[3 * T + 1], H.pos[3 * T + 2], H.pos[3 * T], H.pos[3 * T + 1],
                     H.pos[3 * T + 2]) + P.eps2;
    e_sun -= mass_tar * sqrt(1. / d2);
    d2 = dot3(H.pos[3 * I], H.pos[3 * I + 1], H.pos[3 * I + 2], H.pos[3 * I], H.pos[3 * I + 1],
              H.pos[3 * I + 2]) + P.eps2;
    e_sun -= (mass_imp - 0.) * sqrt(1. / d2);
    e_sun *= P.m_sun;
    // merge_list update
    H.twin_of[I] = jc;
    if (H.flags[I] & GPLUM_FLAG_MERGED) {
        for (int a = 0; a < n; a++) if (H.twin_of[b + a] == ic) H.twin_of[b + a] = jc;
        H.flags[I] &= ~GPLUM_FLAG_MERGED;
    }
    return e_kin + e_int + e_sun;
}

// --------------------------------------------------------------- kernel

// Minimum over the 64 lanes of the wave (every lane active; values not NaN): four DPP
// steps inside each row of 16 lanes, then the four row minima read as scalars.  Far
// shorter latency than a shuffle butterfly through the LDS crossbar.
__device__ inline double wave_min(double v) {
    v = dmin(v, dpp_f64<DPP_QUAD_1032>(v));
    v = dmin(v, dpp_f64<DPP_QUAD_2301>(v));
    v = dmin(v, dpp_f64<DPP_ROW_HALF_MIRROR>(v));
    v = dmin(v, dpp_f64<DPP_ROW_MIRROR>(v));
    return dmin(dmin(readlane_f64(v, 0), readlane_f64(v, 16)), dmin(readlane_f64(v, 32), readlane_f64(v, 48)));
}
// the minimum over each row of 16 lanes, in every lane of the row
__device__ inline double row_min(double v) {
    v = __builtin_fmin(v, dpp_f64<DPP_QUAD_1032>(v));
    v = __builtin_fmin(v, dpp_f64<DPP_QUAD_2301>(v));
    v = __builtin_fmin(v, dpp_f64<DPP_ROW_HALF_MIRROR>(v));
    return __builtin_fmin(v, dpp_f64<DPP_ROW_MIRROR>(v));
}
// Orders the wave's own global-memory writes before its later reads (lane 0 writes
// state that all lanes read back): the wave's memory operations are complete at the
// fence, and the barrier keeps the compiler from moving accesses across it.
__device__ inline void wave_sync() {
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
}

// The active-particle correction of the global-memory path for clusters above HARD_SEQ_MAX
// particles (H.act marks the active ones): the k-th active particle (ascending index)
// goes to wave k mod (waves per workgroup), and the wave's 64 lanes evaluate its hard
// force together (coop_pair_sum); every lane carries the same particle state in
// registers and lane 0 writes it back.  Active particles only read the predicted
// j-data, so the waves need not wait for each other.  Twins of a merged target are
// integrated alongside with their own cut-off radius.
__device__ void coop_correct_active(const HP &P, HardView &H, const JData &J, int b, int n, double t_s,
                                    int flag_col, long long &pairs, int wave, int n_wave) {
    const int32_t *tw = H.twin_of + b;     // cluster-local indices
    const int lane = (int)(threadIdx.x & 63);
    const bool lead = lane == 0;
    int rank = 0;                          // active particles seen so far (wave-uniform)
    for (int i0 = 0; i0 < n; i0 += 64) {
    unsigned long long mask = __ballot(i0 + lane < n && H.act[b + i0 + lane] != 0);
    while (mask) {
        const int i = i0 + __ffsll(mask) - 1;
        mask &= mask - 1;
        if ((rank++) % n_wave != wave) continue;
        const int g = b + i;
        const bool merged = (H.flags[g] & GPLUM_FLAG_MERGED) != 0;
        if (lead) pairs += 3 * (long long)(n - 1);
        // state of g (predicted by the predict pass)
        double xp[3], vp[3], a0s[3], j0s[3], a0d[3], j0d[3], as[3], js[3], ad[3], jd[3];
        double x[3], v[3], a2s[3], a3s[3], a2d[3], a3d[3];
        ld3(H.xp, g, xp); ld3(H.vp, g, vp);
        ld3(H.a0_s, g, a0s); ld3(H.j0_s, g, j0s); ld3(H.a0_d, g, a0d); ld3(H.j0_d, g, j0d);
        const double rinv = H.rinv[g];
        const int64_t id = H.id[g];
        star_acc_jerk(P, xp, vp, as, js, nullptr);
        coop_pair_sum(P, J, n, id, xp, vp, rinv, ad, jd);
        if (merged) {
            // mergeAccJerk over the target and its twins (twin index order)
            double sa[3], sj[3], mass = H.mass[g];
            for (int k = 0; k < 3; k++) { sa[k] = H.mass[g] * ad[k]; sj[k] = H.mass[g] * jd[k]; }
            for (int j = 0; j < n; j++) {
                if (tw[j] != i) continue;
                double txp[3], tvp[3], tad[3], tjd[3], tas[3], tjs[3];
                ld3(H.xp, b + j, txp); ld3(H.vp, b + j, tvp);
                star_acc_jerk(P, txp, tvp, tas, tjs, nullptr);
                coop_pair_sum(P, J, n, H.id[b + j], txp, tvp, H.rinv[b + j], tad, tjd);
                if (lead) { st3(H.acc_s, b + j, tas); st3(H.jerk_s, b + j, tjs); pairs += 3 * (long long)(n - 1); }
                for (int k = 0; k < 3; k++) { sa[k] += H.mass[b + j] * tad[k]; sj[k] += H.mass[b + j] * tjd[k]; }
                mass += H.mass[b + j];
            }
            const double minv = 1. / mass;
            for (int k = 0; k < 3; k++) { ad[k] = sa[k] * minv; jd[k] = sj[k] * minv; }
        }
        const double t_c = t_s - H.time[g];
        for (int ite = 0; ite < 2; ite++) {
            correct_regs(t_c, xp, vp, as, a0s, j0s, js, ad, a0d, j0d, jd, x, v, a2s, a3s, a2d, a3d);
            if (merged && lead)
                for (int j = 0; j < n; j++)
                    if (tw[j] == i) {
                        // the twin's correction from its own predicted state and the merged acc/jerk
                        double txp[3], tvp[3], ta0s[3], tj0s[3], ta0d[3], tj0d[3], tas[3], tjs[3];
                        double tx[3], tv[3], t2s[3], t3s[3], t2d[3], t3d[3];
                        ld3(H.xp, b + j, txp); ld3(H.vp, b + j, tvp);
                        ld3(H.a0_s, b + j, ta0s); ld3(H.j0_s, b + j, tj0s);
                        ld3(H.a0_d, b + j, ta0d); ld3(H.j0_d, b + j, tj0d);
                        ld3(H.acc_s, b + j, tas); ld3(H.jerk_s, b + j, tjs);
                        correct_regs(t_c, txp, tvp, tas, ta0s, tj0s, tjs, ad, ta0d, tj0d, jd, tx, tv, t2s, t3s, t2d,
                                     t3d);
                        st3(H.pos, b + j, tx); st3(H.vel, b + j, tv);
                    }
            wave_sync();
            star_acc_jerk(P, x, v, as, js, nullptr);
            coop_pair_sum(P, J, n, id, x, v, rinv, ad, jd);
            if (merged) {
                double sa[3], sj[3], mass = H.mass[g];
                for (int k = 0; k < 3; k++) { sa[k] = H.mass[g] * ad[k]; sj[k] = H.mass[g] * jd[k]; }
                for (int j = 0; j < n; j++) {
                    if (tw[j] != i) continue;
                    double tx[3], tv[3], tad[3], tjd[3], tas[3], tjs[3];
                    ld3(H.pos, b + j, tx); ld3(H.vel, b + j, tv);
                    star_acc_jerk(P, tx, tv, tas, tjs, nullptr);
                    coop_pair_sum(P, J, n, H.id[b + j], tx, tv, H.rinv[b + j], tad, tjd);
                    wave_sync();
                    if (lead) { st3(H.acc_s, b + j, tas); st3(H.jerk_s, b + j, tjs); }
                    for (int k = 0; k < 3; k++) { sa[k] += H.mass[b + j] * tad[k]; sj[k] += H.mass[b + j] * tjd[k]; }
                    mass += H.mass[b + j];
                }
                const double minv = 1. / mass;
                for (int k = 0; k < 3; k++) { ad[k] = sa[k] * minv; jd[k] = sj[k] * minv; }
            }
        }
        double time = H.time[g] + t_c;
        double dt = H.dt[g];
        if (!flag_col) dt = dt_block(P, time, dt, H.acc0[g], ad, jd, a2d, a3d, as, js, a2s, a3s);
        wave_sync();
        if (lead) {
            st3(H.pos, g, x); st3(H.vel, g, v);
            st3(H.acc_s, g, as); st3(H.jerk_s, g, js); st3(H.acc_d, g, ad); st3(H.jerk_d, g, jd);
            st3(H.a2_s, g, a2s); st3(H.a3_s, g, a3s); st3(H.a2_d, g, a2d); st3(H.a3_d, g, a3d);
            H.time[g] = time;
            if (!flag_col) H.dt[g] = dt;
            if (merged)
                for (int j = 0; j < n; j++)
                    if (tw[j] == i) {
                        st3(H.acc_d, b + j, ad); st3(H.jerk_d, b + j, jd);
                        H.time[b + j] += t_c;
                        if (!flag_col) H.dt[b + j] = dt;
                    }
        }
        wave_sync();
    }
    }
}

// ------------------------------------- global-memory path: workgroup-level reductions

// One slot per wave for each reduction (separate slots, so that a reduction needs no
// barrier before its writes).
struct WaveSlots {
    double ts[8], sys[8], rm[8];
    int lo[8], hi[8];
};

// Minimum over the workgroup (every lane active, values not NaN): the wave's minimum by
// DPP, the waves' minima through slot[] and one barrier.  Exact, hence the value of
// block_min.
__device__ inline double block_min_waves(double v, double *slot) {
    v = wave_min(v);
    if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
    __syncthreads();
    double m = slot[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = dmin(m, slot[w]);
    return m;
}

// (R, lo, hi) lexicographic minimum over the workgroup (every lane active).
__device__ inline bool rlh_less(double r, int lo, int hi, double r2, int lo2, int hi2) {
    return r < r2 || (r == r2 && (lo < lo2 || (lo == lo2 && hi < hi2)));
}
__device__ inline void block_argmin_waves(double &v, int &lo, int &hi, WaveSlots &W) {
    for (int d = 32; d > 0; d >>= 1) {
        const double ov = __shfl_xor(v, d);
        const int ol = __shfl_xor(lo, d), oh = __shfl_xor(hi, d);
        if (rlh_less(ov, ol, oh, v, lo, hi)) { v = ov; lo = ol; hi = oh; }
    }
    if ((threadIdx.x & 63) == 0) {
        const int w = threadIdx.x >> 6;
        W.rm[w] = v; W.lo[w] = lo; W.hi[w] = hi;
    }
    __syncthreads();
    v = W.rm[0]; lo = W.lo[0]; hi = W.hi[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++)
        if (rlh_less(W.rm[w], W.lo[w], W.hi[w], v, lo, hi)) { v = W.rm[w]; lo = W.lo[w]; hi = W.hi[w]; }
}

// After the collision test found the pair (ic, jc) in a block step and the active
// particles were corrected (hermite.h:289-296, 449-458): perfect merging, the full hard
// force of everybody, the merged targets' acc/jerk, the initial block step of the live
// particles and the twins' steps.  Every thread of one workgroup calls it.
__device__ void collision_tail(const HP &P, HardView &H, int b, int n, int ic, int jc, double &ed,
                               long long &pairs) {
    const int t = threadIdx.x;
    const int B = blockDim.x;
    if (t == 0) ed += perfect_merge(P, H, b, n, ic, jc);
    __threadfence_block();
    __syncthreads();
    for (int i = t; i < n; i += B) { gravity_full(P, H, b, n, i); pairs += n - 1; }
    __threadfence_block();
    __syncthreads();
    for (int i = t; i < n; i += B)
        if (H.flags[b + i] & GPLUM_FLAG_MERGED) merge_acc_jerk(H, b, n, i);
    __threadfence_block();
    __syncthreads();
    for (int i = t; i < n; i += B) {
        const int g = b + i;
        if (!(H.flags[g] & GPLUM_FLAG_DEAD)) {
            double ad[3], jd[3], as[3], js[3];
            ld3(H.acc_d, g, ad); ld3(H.jerk_d, g, jd); ld3(H.acc_s, g, as); ld3(H.jerk_s, g, js);
            H.dt[g] = dt_initial(P, H.time[g], H.dt[g], H.acc0[g], ad, jd, as, js);
        }
    }
    __threadfence_block();
    __syncthreads();
    for (int i = t; i < n; i += B)
        if (H.twin_of[b + i] >= 0) H.dt[b + i] = H.dt[b + H.twin_of[b + i]];
    __threadfence_block();
    __syncthreads();
}

// Block steps of a cluster too large for the LDS, from the start of the soft step to its
// end on the global-memory state H (j-data through J), then the final calcGravity.  Every
// thread of the workgroup calls it; collisions and twins handled here.
__device__ void integrate_global(const HP &P, HardView &H, const JData &J, int b, int n, double &sys_time,
                                 long long &loop, double &ed, int &n_col, long long &pairs, WaveSlots &W) {
    const int t = threadIdx.x;
    const int B = blockDim.x;
    const double time_end = P.dt_tree;
    while (sys_time < time_end && loop < BLOCK_STEP_CAP) {
        // makeActiveList: t_s = min(time + dt) over live particles
        double tl = 1.e10;
        for (int i = t; i < n; i += B)
            if (!(H.flags[b + i] & GPLUM_FLAG_DEAD)) tl = dmin(tl, H.time[b + i] + H.dt[b + i]);
        const double t_s = block_min_waves(tl, W.ts);
        // predict all (hermite.h:277-283)
        for (int i = t; i < n; i += B) predict(H, b + i, t_s - H.time[b + i]);
        __threadfence_block();
        __syncthreads();
        // collisionDetermination (hermite.h:98-196)
        int flag_col = 0, ic = -1, jc = -1;
        if (P.collision) {
            double rm = 1.;
            int gi = 0x7fffffff, gj = 0x7fffffff;
            for (int i = t; i < n; i += B) {
                if (H.flags[b + i] & GPLUM_FLAG_DEAD) continue;
                for (int j = 0; j < n; j++) {
                    if (i == j || (H.flags[b + j] & GPLUM_FLAG_DEAD)) continue;
                    const double dx = H.xp[3 * (b + i)] - H.xp[3 * (b + j)];
                    const double dy = H.xp[3 * (b + i) + 1] - H.xp[3 * (b + j) + 1];
                    const double dz = H.xp[3 * (b + i) + 2] - H.xp[3 * (b + j) + 2];
                    const double d2 = dot3(dx, dy, dz, dx, dy, dz);
                    const double r2 = H.f[b + i] * H.r_planet[b + i] + H.f[b + j] * H.r_planet[b + j];
                    if (!(d2 < COL_FILTER * r2 * r2)) continue;
                    const double Rr = sqrt(d2) / r2;
                    if (Rr < rm) { rm = Rr; gi = i; gj = j; }
                }
            }
            block_argmin_waves(rm, gi, gj, W);
            if (rm < 1.) {
                flag_col = 1;
                if (H.mass[b + gi] < H.mass[b + gj]) { ic = gi; jc = gj; } else { ic = gj; jc = gi; }
            }
            if (flag_col)
                for (int i = t; i < n; i += B) H.dt[b + i] = t_s - H.time[b + i];
            __threadfence_block();
            __syncthreads();
        }
        // correct the active particles (hermite.h:300-375)
        for (int i = t; i < n; i += B)
            H.act[b + i] = !(H.flags[b + i] & GPLUM_FLAG_DEAD) &&
                           (flag_col || H.time[b + i] + H.dt[b + i] == t_s);
        __threadfence_block();
        __syncthreads();
        coop_correct_active(P, H, J, b, n, t_s, flag_col, pairs, (int)(threadIdx.x >> 6), B >> 6);
        __threadfence_block();
        __syncthreads();
        if (flag_col) {
            collision_tail(P, H, b, n, ic, jc, ed, pairs);
            n_col++;
        }
        // getSystemTime
        double tm = 1.e10;
        for (int i = t; i < n; i += B)
            if (!(H.flags[b + i] & GPLUM_FLAG_DEAD)) tm = dmin(tm, H.time[b + i]);
        sys_time = block_min_waves(tm, W.sys);
        loop++;
    }
    for (int i = t; i < n; i += B) { gravity_full(P, H, b, n, i); pairs += n - 1; }
    __threadfence_block();
    __syncthreads();
    if (n_col > 0) {
        for (int i = t; i < n; i += B)
            if (H.flags[b + i] & GPLUM_FLAG_MERGED) merge_acc_jerk(H, b, n, i);
    }
    __syncthreads();
}

// ------------------------------------------- clusters of 2 to 4 bodies: lane per term
//
// Lane L = 16 T + 4 q + c works on term T (the rows: T = 0 the Sun, T = k + 1 the pair
// with particle p's k-th partner in ascending index, j = k + (k >= p)), particle p = q
// (the quads of a row; for 2 bodies p = q & 1 and T = (L >> 4) & 1, so that every lane
// holds a copy) and component c (0, 1, 2 = x, y, z; c = 3 pads the quad and keeps
// zeros).  The Sun term and every pair term of every particle are evaluated by the same
// instructions, a vector operation acts on x, y and z at once, and a dot product is the
// quad's sum of its lanes' products in two DPP steps.  Every lane of particle p keeps
// p's state for its component (the same in all rows), so predictor and corrector need
// no exchange; after each evaluation every row gets each row's term of its (p, c) by
// cross-row lane swaps (v_permlane16/32_swap, no LDS) and adds them as star_acc_jerk
// and gravity_loop_lane do (the Sun row; the partner rows in ascending j from zero), and
// the Sun and planet time-step criteria likewise.  Same operations in the same order
// as the reference's loops.

constexpr int DPP_ROW_ROR4 = 0x124;

// (s0 + s1) + s2 on every lane of a quad of lane values s0..s3, which is dot3's sum,
// when the padding value s3 is +0 and s2 is not -0 (squares), or s3 is -0 (any s2):
// s0 + s1 = s1 + s0 and the last addition commute, and s2 + s3 = s2.  All four lanes of
// the quad must be active.
__device__ inline double quad_sum(double s) {
    s = s + dpp_f64<DPP_QUAD_1032>(s);
    return s + dpp_f64<DPP_QUAD_2301>(s);
}
__device__ inline double quad_sq(double a) { return quad_sum(a * a); }
__device__ inline double quad_dot(double a, double b, bool pad) { return quad_sum(pad ? -0. : a * b); }

// Cross-row exchanges.  swap16: each lane gets the values of the even and the odd row
// of its pair of rows (0, 1) or (2, 3), same lane within the row; swap32: the values of
// its half's row at the same position in the lower and the upper half.  Combined, each
// row reads the four rows' values of its lane position.
__device__ inline double dbl_of(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline void swap16(double x, double &even, double &odd) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    even = dbl_of(lo[0], hi[0]);
    odd = dbl_of(lo[1], hi[1]);
}
__device__ inline void swap32(double x, double &low, double &high) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    low = dbl_of(lo[0], hi[0]);
    high = dbl_of(lo[1], hi[1]);
}
// the row values r[0..3] of the lane's position
__device__ inline void rows_of(double x, double (&r)[4]) {
    double lo, hi;
    swap32(x, lo, hi);
    swap16(lo, r[0], r[1]);
    swap16(hi, r[2], r[3]);
}

// Constants of the lane-per-term path.  They are kept in vector registers (the kernel has
// plenty and this path uses few): as scalars the compiler spills and reloads some of them in
// every block step.
struct TermConsts {
    double gamma, g_1_inv, c140, c70, c84, c35, cm20, c3, half_tree, dt_min, alpha2;
    // below the changeover (x < 0, K = 1) at any distance, for the Sun row
    double sun_r_out_inv;
    __device__ explicit TermConsts(const HP &P)
        : gamma(P.cut.gamma), g_1_inv(P.cut.g_1_inv), c140(140.), c70(70.), c84(84.), c35(35.), cm20(-20.), c3(3.),
          half_tree(0.5 * P.dt_tree), dt_min(P.dt_min), alpha2(P.alpha2),
          sun_r_out_inv(P.cut.g_1_inv > 0. ? 1e300 : -1e300) {
        asm("" : "+v"(gamma), "+v"(g_1_inv), "+v"(c140), "+v"(c70), "+v"(c84), "+v"(cm20));
        asm("" : "+v"(c35), "+v"(c3), "+v"(half_tree), "+v"(dt_min), "+v"(alpha2));
    }
};
// The corrector's and predictor's constants of integrate_pair, likewise.
struct StepConsts {
    double third, sixtieth, twelfth, c5, c3a, c6;
    __device__ StepConsts()
        : third(THIRDORDER), sixtieth(ONE_SIXTIETH), twelfth(ONE_TWELFTH), c5(5.), c3a(3. * ALPHA_POS), c6(6.) {
        asm("" : "+v"(third), "+v"(sixtieth), "+v"(twelfth), "+v"(c5), "+v"(c3a), "+v"(c6));
    }
};

// The lane's term of a hard force evaluation (dr = xj - x, d2 = |dr|^2, dv = vj - v), in one instruction stream for the Sun row
// (star_acc_jerk: xj = vj = -0, so that xj - x = -x exactly; mT = m_sun, eps2T =
// eps2_sun) and the partner rows (pair_term with r_out_inv = min of the two 1/r_out):
// the Sun's (1/s, then sqrt) and the pair's (sqrt, then 1/r) sequences are both
// evaluated from one estimate and the row's own one selected.  The Sun row's r_out_inv =
// C.sun_r_out_inv puts it below the changeover (x < 0), so K = 1 and dK/dt is a zero of
// alpha's sign: exact identities (1 K = K, alpha 1 = alpha, 3 alpha + 0 = 3 alpha) that leave
// star_acc_jerk's acc = mj dr and jerk = mj (dv - 3 alpha dr).  need: the lane's term is used.
__device__ inline void term_eval(const TermConsts &C, bool sun, bool pad, bool need, double dr, double d2, double dv,
                                 double mT, double eps2T, double r_out_inv, double &ta, double &tj) {
    const double s = d2 + eps2T;
    // y1: the Sun's 1/r^2, the pair's r
    double y1, rinv, r2inv;
    {
        double g, h;
        root_seed(s, g, h);
        const double y = 2. * h;
        const double a = rcp_fix(s, y * y), b = root_fix(s, g, h);
        const double c = root_fix(a, y, 0.5 * g), d = rcp_fix(b, y);
        y1 = sun ? a : b;
        rinv = sun ? c : d;
        r2inv = sun ? a : d * d;
    }
    if (__ballot(need && (!root_range(s) || rcp_exception(sun ? s : y1)))) {
        const double a = 1. / s, b = sqrt(s);
        y1 = sun ? a : b;
        const double c = sqrt(y1), d = 1. / y1;
        rinv = sun ? c : d;
        r2inv = sun ? y1 : d * d;
    }
    const double r3inv = r2inv * rinv;
    const double mj_r3 = mT * r3inv;
    const double alpha = quad_dot(dr, dv, pad) * r2inv;
    // cutoff_K_sel and cutoff_dKdt_sel
    const double x = (C.gamma - y1 * r_out_inv) * C.g_1_inv;
    const double x2 = x * x, x_1 = x - 1.;
    const double poly = (((C.cm20 * x + C.c70) * x - C.c84) * x + C.c35) * x2 * x2;
    const double slope = C.c140 * x * x * x * x_1 * x_1 * x_1 * r_out_inv * C.g_1_inv;
    const bool below = x < 0., above = x >= 1.;
    const double K = 1. - (below ? 0. : (above ? 1. : poly));
    const double dKdt = alpha * y1 * ((below || above) ? 0. : slope);
    const double alpha_c = alpha * K;
    const double c2 = C.c3 * alpha_c + dKdt;
    ta = mj_r3 * K * dr;
    tj = mj_r3 * (K * dv - c2 * dr);
}

// Every row of particle p gets the Sun term and the sum of the partner terms of its
// component (rows 1..N-1, added in ascending j from zero).
template <int N>
__device__ inline void gather_terms(double ta, double tj, double &as, double &js, double &ad, double &jd) {
    double ra[4], rj[4];
    rows_of(ta, ra);
    rows_of(tj, rj);
    as = ra[0];
    js = rj[0];
    ad = 0.;
    jd = 0.;
#pragma unroll
    for (int k = 1; k < N; k++) {
        ad += ra[k];
        jd += rj[k];
    }
}

// predict_regs and correct_regs for one component (same expressions).
__device__ inline void predict_one(double Dt, double pos, double vel, double as, double js, double ad, double jd,
                                   double &xp, double &vp) {
    const double acc_sd = as + ad;
    const double jerk_sd = js + jd;
    xp = pos + Dt * (vel + Dt * (SECONDORDER * acc_sd + THIRDORDER * Dt * jerk_sd));
    vp = vel + Dt * (acc_sd + Dt * SECONDORDER * jerk_sd);
}
__device__ inline void correct_one(double Dt, double Dt2, double Dt_inv2, double Dt_inv3, double xp, double vp,
                                   double as, double a0s, double j0s, double js, double ad, double a0d, double j0d,
                                   double jd, double &pos, double &vel, double &a2s, double &a3s, double &a2d,
                                   double &a3d) {
    const double Am_s = as - a0s;
    const double J0_s = Dt * j0s;
    const double J1_s = Dt * js;
    const double A2_s = 3. * Am_s - (J1_s + 2. * J0_s);
    const double A3_s = -2. * Am_s + (J1_s + J0_s);
    a2s = 2. * Dt_inv2 * (A2_s + 3. * A3_s);
    a3s = 6. * Dt_inv3 * A3_s;
    const double Am_d = ad - a0d;
    const double J0_d = j0d * Dt;
    const double J1_d = jd * Dt;
    const double A2_d = 3. * Am_d - (J1_d + 2. * J0_d);
    const double A3_d = -2. * Am_d + (J1_d + J0_d);
    a2d = 2. * (A2_d + 3. * A3_d) * Dt_inv2;
    a3d = 6. * A3_d * Dt_inv3;
    const double A2_sd = A2_s + A2_d;
    const double A3_sd = A3_s + A3_d;
    pos = xp + ONE_SIXTIETH * Dt2 * (5. * A2_sd + 3. * ALPHA_POS * A3_sd);
    vel = vp + ONE_TWELFTH * Dt * (4. * A2_sd + 3. * A3_sd);
}

// calc_dt4_fast and calc_dt4 of the lane's term (the row's vectors, dots over the quad).  The
// fast one gives NaN whenever a product is not normal.
__device__ inline double dt4_fast_quad(double eta, double alpha2, double acc0, double a, double j, double s,
                                       double c) {
    const double Acc2 = quad_sq(a) + alpha2 * acc0 * acc0;
    const double Jerk2 = quad_sq(j);
    const double Snap2 = quad_sq(s);
    const double Crac2 = quad_sq(c);
    const double as2 = Acc2 * Snap2, jc2 = Jerk2 * Crac2;
    const double num = __builtin_amdgcn_sqrt(as2) + Jerk2;
    const double den = __builtin_amdgcn_sqrt(jc2) + Snap2;
    const double q = eta * __builtin_amdgcn_sqrt(num * __builtin_amdgcn_rcp(den));
    return (Jerk2 > 0.) ? (__builtin_fmin(as2, jc2) >= DBL_MIN ? q : __builtin_nan("")) : DBL_MAX;
}
__device__ inline double dt4_quad(double eta, double alpha2, double acc0, double a, double j, double s, double c) {
    const double Acc = sqrt(quad_sq(a) + alpha2 * acc0 * acc0);
    const double Jerk2 = quad_sq(j);
    const double Jerk = sqrt(Jerk2);
    const double Snap2 = quad_sq(s);
    const double Snap = sqrt(Snap2);
    const double Crac = sqrt(quad_sq(c));
    return (Jerk > 0.) ? eta * sqrt((Acc * Snap + Jerk2) / (Jerk * Crac + Snap2)) : DBL_MAX;
}

// the Sun row's and the first partner row's values of the lane's position
template <int N>
__device__ inline void sun_planet_of(double x, double &f_sun, double &f_planet) {
    if (N == 2) {
        swap16(x, f_sun, f_planet);
    } else {
        double lo, hi;
        swap32(x, lo, hi);
        swap16(lo, f_sun, f_planet);
    }
}

// dt_block with the Sun criterion from the Sun row and the planet criterion from the
// partner rows (each lane evaluates its own row's, reads the other by a lane swap); the
// exact criteria when either fast one is not finite or dt_1 lies near the step grid.
// DYADIC: the cluster's steps, dt_tree and dt_min are powers of two and its
// times whole multiples of its steps (dyadic_steps), so the largest step that divides time is
// min(2 dt, dt_tree / 2) or dt, the halvings end at min(that, max(the power of two at or below
// dt_1, dt / 2)), and a step below 2 dt_min is at most dt_min.
__device__ inline double hi_word(int hi) { return __longlong_as_double((long long)((unsigned long long)(unsigned)hi << 32)); }
__device__ inline int hi_of(double d) { return (int)(__double_as_longlong(d) >> 32); }
template <int N, bool DYADIC>
__device__ inline double dt_block_rows(const TermConsts &C, double time, double dt, double etaT, double acc0T,
                                       double a, double j, double s, double c) {
    const double dt_max = __builtin_fmin(2. * dt, C.half_tree);
    double dt_0;
    bool cap = false;
    if (DYADIC) {
        const double q = time * hi_word(0x7FE00000 - hi_of(dt_max));
        dt_0 = (q == floor(q)) ? dt_max : dt;
    } else {
        dt_0 = dt_candidate(time, dt_max, cap);
    }
    double f_sun, f_planet;
    sun_planet_of<N>(dt4_fast_quad(etaT, C.alpha2, acc0T, a, j, s, c), f_sun, f_planet);
    double dt_1 = dmin(f_planet, f_sun);
    const unsigned hi = (unsigned)hi_of(dt_1);
    bool clear = (hi & 0xFFFFFu) - 1025u < 0x100000u - 2049u - 1025u && hi - (24u << 20) <= (1998u << 20);
    if (!DYADIC) clear = clear_of_grid(dt_1, dt_0);
    const bool exact = !(f_planet <= DBL_MAX && f_sun <= DBL_MAX && clear);
    if (__ballot(exact)) {
        double e_sun, e_planet;
        sun_planet_of<N>(dt4_quad(etaT, C.alpha2, acc0T, a, j, s, c), e_sun, e_planet);
        if (exact) dt_1 = dmin(e_planet, e_sun);
    }
    if (!DYADIC) {
        const double d = dt_reduce(dt_0, dt_1, dt);
        return (cap || d < 2. * C.dt_min) ? C.dt_min : d;
    }
    const double low = __builtin_fmax(hi_word(hi_of(dt_1) & 0x7FF00000), 0.5 * dt);
    return __builtin_fmax(__builtin_fmin(dt_0, low), C.dt_min);
}

// Whether a particle's starting state keeps to dt_block_rows' dyadic rule, dt_tree and dt_min
// being powers of two no more than 2^50 apart (dyadic_tree).
__device__ inline bool dyadic_steps(const HP &P, double time, double dt) {
    const double q = time * pow2_inverse(dt);
    return is_pow2(dt) && dt >= P.dt_min && time >= 0. && time <= P.dt_tree && q == floor(q);
}
static bool dyadic_tree(const gplum_params &p) {
    return is_pow2(p.dt_tree) && is_pow2(p.dt_min) && p.dt_min <= 0.5 * p.dt_tree && p.dt_min >= 0x1p-50 * p.dt_tree;
}
bool hard_off_grid(const gplum_params &p, double dt) { return dyadic_tree(p) && !(is_pow2(dt) && dt >= p.dt_min); }

// The end of integrate_terms and integrate_pair: the final calcGravity with potentials
// (hermite.h:466-470), one lane per particle.  vec: the lane holds component c of particle p's
// x and v; lead: its time and dt.
template <int N>
__device__ inline void terms_finish(const HP &P, HardView &H, const JData &J, double *s_x, double *s_v, const double *s_ri,
                                    double *s_tm, int b, int p, int c, bool vec, bool lead, double x,
                                    double v, double time, double dt, long long &pairs) {
    const int L = threadIdx.x;
    __syncthreads();
    if (vec) {
        s_x[3 * p + c] = x;
        s_v[3 * p + c] = v;
    }
    if (lead) {
        s_tm[2 * p] = time;
        s_tm[2 * p + 1] = dt;
    }
    __syncthreads();
    if (L < N) {
        const int gi = b + L;
        double xi[3], vi[3], fas[3], fjs[3], fad[3], fjd[3], phs = 0., phd = 0.;
        ld3(s_x, L, xi);
        ld3(s_v, L, vi);
        star_acc_jerk(P, xi, vi, fas, fjs, &phs);
        gravity_loop_lane(P, J, N, L, xi, vi, s_ri[L], fad, fjd, &phd);
        pairs += N - 1;
        st3(H.pos, gi, xi); st3(H.vel, gi, vi);
        st3(H.acc_s, gi, fas); st3(H.jerk_s, gi, fjs);
        st3(H.acc_d, gi, fad); st3(H.jerk_d, gi, fjd);
        H.time[gi] = s_tm[2 * L];
        H.dt[gi] = s_tm[2 * L + 1];
        H.phi_s[gi] = phs;
        H.phi_d[gi] = phd;
        H.flags[gi] &= ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
        H.twin_of[gi] = -1;
    }
    __syncthreads();
}

// Block steps of a cluster of N (3 or 4) particles with distinct ids from the start of the
// soft step (the layout above; one wave; DYADIC: all of them keep to dyadic_steps).  Returns
// false when a block step may have a collision: the state of the start of that block step is
// then in H (flags and twins cleared) for integrate_seq.  Else the final calcGravity with
// potentials is done and written to H.  s_m, s_ri, s_fr hold the cluster's masses, 1/r_out
// and f r_planet; s_x, s_v and s_tm are free.
template <int N, bool DYADIC>
__device__ bool integrate_terms(const HP &P, HardView &H, const JData &J, double *s_x, double *s_v, double *s_m,
                                double *s_ri, double *s_fr, double *s_tm, int b, double &sys_time,
                                long long &loop, long long &pairs) {
    constexpr int m = N - 1;
    const int L = threadIdx.x;
    const int T = L >> 4, p = (L >> 2) & 3;
    const int c = L & 3;
    // lanes of a particle: every row takes part in the evaluations, so that the cross-row
    // swaps read computed values (rows T >= N, 3 bodies, evaluate a don't-care term)
    const bool own = p < N;
    const bool row = own && T < N;                  // lanes of a term of a particle
    const bool sun = T == 0, pad = c == 3;
    const int j = (T >= 1) ? (T - 1) + ((T - 1) >= p ? 1 : 0) : p;   // the row's partner
    const int jc = (j < N) ? j : 0, pc = own ? p : 0;
    const int g = b + pc;
    const TermConsts C(P);
    const double mT = sun ? P.m_sun : s_m[jc];
    const double eps2T = sun ? P.eps2_sun : P.eps2;
    const double r_out_inv = sun ? C.sun_r_out_inv : dmin(s_ri[pc], s_ri[jc]);
    const double etaT = sun ? P.eta_sun : P.eta;
    const double r2c = s_fr[pc] + s_fr[jc];
    const double col_thr = COL_FILTER * r2c * r2c;
    const bool col_row = P.collision && row && !sun;
    const int src = 4 * jc + c;                     // a lane of the partner's component
    const double time_end = P.dt_tree;
    double x = 0., v = 0., time = 0., dt = 0., acc0 = 0.;
    if (own && !pad) {
        x = H.pos[3 * g + c];
        v = H.vel[3 * g + c];
    }
    if (own) {
        time = H.time[g];
        dt = H.dt[g];
        acc0 = H.acc0[g];
    }
    const double acc0T = sun ? 0. : acc0;
    const bool lead = row && sun && c == 0;
    double as = 0., js = 0., ad = 0., jd = 0., a2s = 0., a3s = 0., a2d = 0., a3d = 0.;
    {
        // initial calcGravity (hermite.h:259-270) at the current state
        double xj = __shfl(x, src), vj = __shfl(v, src);
        if (sun) { xj = -0.; vj = -0.; }
        if (own) {
            double ta, tj;
            const double dr = xj - x;
            term_eval(C, sun, pad, row, dr, quad_sq(dr), vj - v, mT, eps2T, r_out_inv, ta, tj);
            gather_terms<N>(ta, tj, as, js, ad, jd);
        }
    }
    // the smallest value of the particles (quads of a row)
    auto smallest = [](double u) __attribute__((always_inline)) {
        u = __builtin_fmin(u, dpp_f64<DPP_ROW_ROR4>(u));
        u = __builtin_fmin(u, dpp_f64<DPP_ROW_ROR8>(u));
        return readlane_f64(u, 0);
    };
    double t_s = smallest(own ? time + dt : 1.e10);
    bool handover = false;
    while (sys_time < time_end && loop < BLOCK_STEP_CAP) {
        const double Dt = t_s - time;
        const double a0s = as, j0s = js, a0d = ad, j0d = jd;
        double xp = 0., vp = 0.;
        predict_one(Dt, x, v, as, js, ad, jd, xp, vp);
        double xj = __shfl(xp, src), vj = __shfl(vp, src);
        if (sun) { xj = -0.; vj = -0.; }
        // collisionDetermination: a pair with R = |dr| / (f_i R_i + f_j R_j) < 1; R itself is left
        // to integrate_seq
        const double drp = xj - xp, d2p = quad_sq(drp);
        if (__ballot(col_row && d2p < col_thr)) { handover = true; break; }
        if (own && time + dt == t_s) {
            if (lead) pairs += 3 * (long long)m;
            const double Dt2 = Dt * Dt;
            // DYADIC: Dt = dt, a power of two
            const double Dt_inv = DYADIC ? hi_word(0x7FE00000 - hi_of(Dt)) : recip_step(Dt);
            const double Dt_inv2 = Dt_inv * Dt_inv;
            const double Dt_inv3 = Dt_inv2 * Dt_inv;
            double ta, tj;
            term_eval(C, sun, pad, row, drp, d2p, vj - vp, mT, eps2T, r_out_inv, ta, tj);
            gather_terms<N>(ta, tj, as, js, ad, jd);
            for (int ite = 0; ite < 2; ite++) {
                correct_one(Dt, Dt2, Dt_inv2, Dt_inv3, xp, vp, as, a0s, j0s, js, ad, a0d, j0d, jd, x, v, a2s, a3s,
                            a2d, a3d);
                const double dr = xj - x;
                term_eval(C, sun, pad, row, dr, quad_sq(dr), vj - v, mT, eps2T, r_out_inv, ta, tj);
                gather_terms<N>(ta, tj, as, js, ad, jd);
            }
            time += Dt;
            dt = dt_block_rows<N, DYADIC>(C, time, dt, etaT, acc0T, sun ? as : ad, sun ? js : jd, sun ? a2s : a2d,
                                  sun ? a3s : a3d);
        }
        // the system time is asked for once the next block time has reached the end: before
        // that some particle's time is below it
        t_s = smallest(own ? time + dt : 1.e10);
        if (!(t_s < time_end)) sys_time = smallest(own ? time : 1.e10);
        loop++;
    }
    if (handover) {
        // the state at the start of this block step, for integrate_seq
        if (row && sun && !pad) {
            H.pos[3 * g + c] = x; H.vel[3 * g + c] = v;
            H.acc_s[3 * g + c] = as; H.jerk_s[3 * g + c] = js;
            H.acc_d[3 * g + c] = ad; H.jerk_d[3 * g + c] = jd;
        }
        if (lead) {
            H.time[g] = time;
            H.dt[g] = dt;
            H.flags[g] &= ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
            H.twin_of[g] = -1;
        }
        return false;
    }
    terms_finish<N>(P, H, J, s_x, s_v, s_ri, s_tm, b, p, c, row && sun && !pad, lead, x, v, time, dt, pairs);
    return true;
}

// integrate_terms for two bodies, whose chain bounds most soft steps (the cluster with the most
// block steps is nearly always a pair): row T keeps only its own term's acc and jerk (Sun or
// partner) and their derivatives, and the rows are added where the predictor and the corrector
// add them (as + ad, A2_s + A2_d, ...), so the corrector is evaluated once for both.  Bound by
// instruction issue of its one wave (560 per block step of 4 cycles; 606 when every row kept both
// terms: 2 bodies 1.06 us per block step in a 100k disk).
template <bool DYADIC>
__device__ bool integrate_pair(const HP &P, HardView &H, const JData &J, double *s_x, double *s_v, double *s_m,
                               double *s_ri, double *s_fr, double *s_tm, int b, double &sys_time,
                               long long &loop, long long &pairs) {
    const int L = threadIdx.x;
    const int T = (L >> 4) & 1, p = (L >> 2) & 1, c = L & 3;
    const bool sun = T == 0, pad = c == 3;
    const bool first = L < 32 && ((L >> 2) & 3) < 2;             // not a copy
    const int g = b + p;
    const TermConsts C(P);
    const StepConsts K;
    const double mT = sun ? P.m_sun : s_m[1 - p];
    const double eps2T = sun ? P.eps2_sun : P.eps2;
    const double r_out_inv = sun ? C.sun_r_out_inv : dmin(s_ri[p], s_ri[1 - p]);
    const double etaT = sun ? P.eta_sun : P.eta;
    // the partner's term is added to zero (gravity_loop_lane), the Sun's is not: + -0 changes nothing
    const double zero = sun ? -0. : 0.;
    const double r2c = s_fr[0] + s_fr[1];
    const double col_thr = (P.collision && !sun) ? COL_FILTER * r2c * r2c : -1.;
    const double time_end = P.dt_tree;
    double x = pad ? 0. : H.pos[3 * g + c], v = pad ? 0. : H.vel[3 * g + c];
    double time = H.time[g], dt = H.dt[g];
    const double acc0T = sun ? 0. : H.acc0[g];
    const bool lead = sun && c == 0 && first;
    // the partner is the next quad (quads 2, 3 are copies of 0, 1)
    auto partner = [&](double u) __attribute__((always_inline)) { return sun ? -0. : dpp_f64<DPP_ROW_ROR4>(u); };
    auto both = [](double u) __attribute__((always_inline)) {
        double even, odd;
        swap16(u, even, odd);
        return even + odd;
    };
    auto smallest = [](double u) __attribute__((always_inline)) {
        return readlane_f64(__builtin_fmin(u, dpp_f64<DPP_ROW_ROR4>(u)), 0);
    };
    double a, j, a2 = 0., a3 = 0.;
    auto force = [&](double dr, double d2, double dv) __attribute__((always_inline)) {
        double ta, tj;
        term_eval(C, sun, pad, true, dr, d2, dv, mT, eps2T, r_out_inv, ta, tj);
        a = ta + zero;
        j = tj + zero;
    };
    {
        // initial calcGravity (hermite.h:259-270) at the current state
        const double dr = partner(x) - x;
        force(dr, quad_sq(dr), partner(v) - v);
    }
    double t_next = time + dt;
    double t_s = smallest(t_next);
    bool handover = false;
    int n_eval = 0;
    while (sys_time < time_end && loop < BLOCK_STEP_CAP) {
        const double Dt = t_s - time;
        const double acc_sd = both(a), jerk_sd = both(j);
        const double xp = x + Dt * (v + Dt * (SECONDORDER * acc_sd + K.third * Dt * jerk_sd));
        const double vp = v + Dt * (acc_sd + Dt * SECONDORDER * jerk_sd);
        const double xj = partner(xp), vj = partner(vp);
        // collisionDetermination: R = |dr| / (f_i R_i + f_j R_j) < 1; R itself is left to
        // integrate_seq
        const double drp = xj - xp, d2p = quad_sq(drp);
        if (__ballot(d2p < col_thr)) { handover = true; break; }
        if (t_next == t_s) {
            n_eval++;
            const double Dt2 = Dt * Dt;
            // DYADIC: Dt = dt, a power of two
            const double Dt_inv = DYADIC ? hi_word(0x7FE00000 - hi_of(Dt)) : recip_step(Dt);
            const double Dt_inv2 = Dt_inv * Dt_inv, Dt_inv3 = Dt_inv2 * Dt_inv;
            const double a0 = a, J0 = Dt * j;
            force(drp, d2p, vj - vp);
            for (int ite = 0; ite < 2; ite++) {
                const double Am = a - a0;
                const double J1 = Dt * j;
                const double A2 = C.c3 * Am - (J1 + 2. * J0);
                const double A3 = -2. * Am + (J1 + J0);
                a2 = 2. * Dt_inv2 * (A2 + C.c3 * A3);
                a3 = K.c6 * Dt_inv3 * A3;
                if (!DYADIC && !sun) a3 = K.c6 * A3 * Dt_inv3;
                const double A2_sd = both(A2), A3_sd = both(A3);
                x = xp + K.sixtieth * Dt2 * (K.c5 * A2_sd + K.c3a * A3_sd);
                v = vp + K.twelfth * Dt * (4. * A2_sd + C.c3 * A3_sd);
                const double dr = xj - x;
                force(dr, quad_sq(dr), vj - v);
            }
            time += Dt;
            dt = dt_block_rows<2, DYADIC>(C, time, dt, etaT, acc0T, a, j, a2, a3);
            t_next = time + dt;
        }
        // the system time is asked for once the next block time has reached the end: before
        // that some particle's time is below it
        t_s = smallest(t_next);
        if (!(t_s < time_end)) sys_time = smallest(time);
        loop++;
    }
    if (lead) pairs += 3 * (long long)n_eval;
    if (handover) {
        // the state at the start of this block step, for integrate_seq
        if (!pad && first) {
            if (sun) { H.pos[3 * g + c] = x; H.vel[3 * g + c] = v; }
            (sun ? H.acc_s : H.acc_d)[3 * g + c] = a;
            (sun ? H.jerk_s : H.jerk_d)[3 * g + c] = j;
        }
        if (lead) {
            H.time[g] = time;
            H.dt[g] = dt;
            H.flags[g] &= ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
            H.twin_of[g] = -1;
        }
        return false;
    }
    terms_finish<2>(P, H, J, s_x, s_v, s_ri, s_tm, b, p, c, sun && !pad && first, lead, x, v, time, dt, pairs);
    return true;
}

}  // namespace gplum

#include "hermite_lds.hpp"

namespace gplum {

// The clusters of a launch, pulled from a queue (persistent) or one per workgroup: calls
// run(c, b, n, sys_time, loop, ed, n_col, pairs) for those of lo < n <= hi members and
// records the outcome.  Every thread of the workgroup calls it.
template <class F>
__device__ __forceinline__ void cluster_queue(const HP &P, const ClusterArgs &A, int lo, int hi, F run) {
    __shared__ int s_cl;
    __shared__ unsigned long long s_pairs;
    const int t = threadIdx.x;
    const int B = blockDim.x;
    for (int iter = 0;; iter++) {
        if (t == 0) s_cl = A.persistent ? atomicAdd(A.next, 1) : ((iter == 0) ? (int)blockIdx.x : A.ncl);
        __syncthreads();
        const int q = s_cl;
        __syncthreads();
        if (q >= A.ncl) break;
        const int c = A.order ? A.order[q] : q;
        const int b = __builtin_amdgcn_readfirstlane(A.off[c]);
        const int n = __builtin_amdgcn_readfirstlane(A.off[c + 1]) - b;
        if (n <= lo || n > hi) continue;
        // pair evaluations of this cluster (hard_pair calls), for the roofline: those of the
        // initial calcGravity first
        long long pairs = (long long)(n - 1) * ((t < n) ? (n - 1 - t) / B + 1 : 0);
        if (t == 0) s_pairs = 0ull;
        double ed = 0.;
        int n_col = 0;
        long long loop = 0;
        double sys_time = 0.;
        run(b, n, sys_time, loop, ed, n_col, pairs);
        __syncthreads();
        atomicAdd(&s_pairs, (unsigned long long)pairs);
        __syncthreads();
        if (t == 0) {
            A.edisp[c] = ed;
            A.ncol[c] = n_col;
            A.nblock[c] = (sys_time < P.dt_tree) ? -1 : loop;   // -1: block-step cap reached
            A.npair[c] = (long long)s_pairs;
        }
        __syncthreads();
    }
}

// Clusters of up to HERMITE_SMALL members, one wave each: 2 to terms_max bodies with a lane
// per term (a collision hands over to the LDS path in the middle of the soft step), the
// others on the LDS path.  The arguments are read from LDS: in scalar registers they would
// be spilled and reloaded in the block-step loop.  DYADIC: dyadic_tree's parameters, as in
// every ordinary run; a cluster whose own steps are not powers of two then takes the LDS path
// (hard_launch gives those that its caller lists to the other instantiation).
template <bool DYADIC>
__global__ __launch_bounds__(HERMITE_BLOCK) void k_hermite_small(HP P_arg, HardView H_arg, ClusterArgs A_arg, int lo,
                                                                 int hi) {
    __shared__ HP P;
    __shared__ HardView H;
    __shared__ ClusterArgs A;
    __shared__ ClusterLds<HERMITE_SMALL> C;
    constexpr int TP = lds_terms(HERMITE_BLOCK, 1, HERMITE_SMALL);
    __shared__ double2 s_term[3 * TP];
    const int t = threadIdx.x;
    if (t == 0) {
        P = P_arg;
        H = H_arg;
        A = A_arg;
    }
    __syncthreads();
    cluster_queue(P, A, lo, hi, [&](int b, int n, double &sys_time, long long &loop, double &ed, int &n_col,
                                    long long &pairs) {
        bool fresh = true;
        if (n >= 2 && n <= P.terms_max) {
            if (t < n) {
                C.mass[t] = H.mass[b + t];
                C.rinv[t] = H.rinv[b + t];
                C.id[t] = H.id[b + t];
                C.fr[t] = H.f[b + t] * H.r_planet[b + t];
            }
            __syncthreads();
            // the clusters the reference forms have distinct ids, and the lane-per-term path
            // leaves the id test out
            bool other = false;
            if (t < n) {
                other = DYADIC && !dyadic_steps(P, H.time[b + t], H.dt[b + t]);
                for (int j = 0; j < n; j++) other = other || (j != t && C.id[j] == C.id[t]);
            }
            if (__ballot(other) == 0) {
                const JData J{C.xp, C.vp, C.mass, C.rinv, C.id};
                double *tm = reinterpret_cast<double *>(s_term);
                auto terms = [&](auto N) {
                    return integrate_terms<N.value, DYADIC>(P, H, J, C.xp, C.vp, C.mass, C.rinv, C.fr, tm, b, sys_time,
                                                            loop, pairs);
                };
                const bool done = (n == 2) ? integrate_pair<DYADIC>(P, H, J, C.xp, C.vp, C.mass, C.rinv, C.fr, tm, b,
                                                                    sys_time, loop, pairs)
                                  : (n == 3) ? terms(std::integral_constant<int, 3>())
                                             : terms(std::integral_constant<int, 4>());
                if (done) return;
                fresh = false;
                __threadfence_block();
                __syncthreads();
            }
        }
        run_cluster_lds<HERMITE_SMALL, HERMITE_BLOCK>(P, H, C, b, n, fresh, n_col, pairs, [&](HardView &V) {
            integrate_seq<HERMITE_SMALL, HERMITE_BLOCK, TP>(P, C, V, s_term, n, sys_time, loop, ed, n_col, pairs);
        });
    });
}

// Clusters of NMIN to NMAX <= HARD_SEQ_MAX members on T threads.
// (two waves per SIMD: two to four clusters of a large batch share a CU)
template <int NMIN, int NMAX, int T>
__global__ __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(2))) void k_hermite_mid(HP P, HardView H_arg, ClusterArgs A_arg, int lo, int hi) {
    __shared__ HardView H;
    __shared__ ClusterArgs A;
    __shared__ ClusterLds<NMAX> C;
    constexpr int TP = lds_terms(T, NMIN, NMAX);
    __shared__ double2 s_term[3 * TP];
    if (threadIdx.x == 0) {
        H = H_arg;
        A = A_arg;
    }
    __syncthreads();
    cluster_queue(P, A, lo, hi, [&](int b, int n, double &sys_time, long long &loop, double &ed, int &n_col,
                                    long long &pairs) {
        run_cluster_lds<NMAX, T>(P, H, C, b, n, true, n_col, pairs, [&](HardView &V) {
            integrate_seq<NMAX, T, TP>(P, C, V, s_term, n, sys_time, loop, ed, n_col, pairs);
        });
    });
}

// Clusters of HARD_SEQ_MAX + 1 to HERMITE_LDS members.
__global__ __launch_bounds__(HERMITE_BIG_BLOCK) void k_hermite_big(HP P, HardView H_arg, ClusterArgs A_arg, int lo,
                                                                   int hi) {
    __shared__ HardView H;
    __shared__ ClusterArgs A;
    __shared__ ClusterLds<HERMITE_LDS> C;
    __shared__ TreeLds<HERMITE_LDS> E;
    if (threadIdx.x == 0) {
        H = H_arg;
        A = A_arg;
    }
    __syncthreads();
    cluster_queue(P, A, lo, hi, [&](int b, int n, double &sys_time, long long &loop, double &ed, int &n_col,
                                    long long &pairs) {
        run_cluster_lds<HERMITE_LDS, HERMITE_BIG_BLOCK>(P, H, C, b, n, true, n_col, pairs, [&](HardView &V) {
            integrate_tree<HERMITE_LDS, HERMITE_BIG_BLOCK>(P, C, E, V, n, sys_time, loop, ed, n_col, pairs);
        });
    });
}

// Larger clusters on the global-memory state: eight waves, two per SIMD (256 registers per
// lane).
__global__ __launch_bounds__(HERMITE_GLOBAL_BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_hermite_global(
    HP P, HardView H, ClusterArgs A, int lo, int hi) {
    __shared__ WaveSlots W;
    const int t = threadIdx.x;
    cluster_queue(P, A, lo, hi, [&](int b, int n, double &sys_time, long long &loop, double &ed, int &n_col,
                                    long long &pairs) {
        const JData J{H.xp + 3 * b, H.vp + 3 * b, H.mass + b, H.rinv + b, H.id + b};
        // initial calcGravity for all, flags cleared (hermite.h:259-270)
        for (int i = t; i < n; i += HERMITE_GLOBAL_BLOCK) {
            gravity_full(P, H, b, n, i);
            H.flags[b + i] &= ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
            H.twin_of[b + i] = -1;
        }
        __threadfence_block();
        __syncthreads();
        integrate_global(P, H, J, b, n, sys_time, loop, ed, n_col, pairs, W);
    });
}

// ------------------------------------------------------------- isolated

// timeIntegrateKepler_isolated (hermite.h:787-815) / timeIntegrate_isolated
// (hermite.h:734-785) chosen as in hard.h:803-811.
struct IsoView {
    double *pos, *vel, *acc_d, *jerk_d, *acc_s, *jerk_s, *phi_d, *phi_s, *time, *dt, *acc0;
    const int32_t *number;
    int32_t *n_cluster;
};

__device__ double solve_kepler(double l, double ecc) {
    const double ecc2 = ecc * ecc, ecc3 = ecc2 * ecc, ecc4 = ecc2 * ecc2, ecc5 = ecc3 * ecc2, ecc6 = ecc3 * ecc3;
    double u = l + (ecc - ecc3 / 8. + ecc5 / 192.) * sin(l) + (ecc2 / 2. - ecc4 / 6. + ecc6 / 48.) * sin(2. * l) +
               (3. * ecc3 / 8. - 27. * ecc5 / 128.) * sin(3. * l) + (ecc4 / 3. - 4. * ecc6 / 15.) * sin(4. * l) +
               125. * ecc5 / 384. * sin(5. * l) + 27. * ecc6 / 80. * sin(6. * l);
    if (fabs((u - ecc * sin(u)) - l) > 1.e-15) {
        double u0;
        int loop = 0;
        do {
            u0 = u;
            const double s = sin(u0), c = cos(u0);
            u = u0 - ((u0 - ecc * s - l) / (1. - ecc * c));
            loop++;
        } while (fabs(u - u0) > 1.e-15 && loop < 10);
    }
    return u;
}

__device__ inline double eccentricity(const HP &P, const double x[3], const double v[3]) {
    const double r = sqrt(dot3(x[0], x[1], x[2], x[0], x[1], x[2]));
    const double rv = dot3(x[0], x[1], x[2], v[0], v[1], v[2]);
    const double ax = 1.0 / (2.0 / r - dot3(v[0], v[1], v[2], v[0], v[1], v[2]) / P.m_sun);
    const double ecccosu = 1. - r / ax;
    const double eccsinu2 = rv * rv / (P.m_sun * ax);
    return sqrt(ecccosu * ecccosu + eccsinu2);
}

__device__ void kepler_drift(const HP &P, double x[3], double v[3], double dtime) {
    const double mu = P.m_sun;
    const double r = sqrt(dot3(x[0], x[1], x[2], x[0], x[1], x[2]));
    const double rinv = 1. / r;
    const double v2 = dot3(v[0], v[1], v[2], v[0], v[1], v[2]);
    const double rv = dot3(x[0], x[1], x[2], v[0], v[1], v[2]);
    const double ax = 1.0 / (2.0 * rinv - v2 / mu);
    const double ecccosu = 1. - r / ax;
    const double eccsinu = rv / sqrt(mu * ax);
    const double ecc = sqrt(ecccosu * ecccosu + eccsinu * eccsinu);
    const double nn = sqrt(mu / (ax * ax * ax));
    double u, cosu, sinu;
    if (ecc != 0) { u = atan2(eccsinu, ecccosu); cosu = ecccosu / ecc; sinu = eccsinu / ecc; }
    else { u = 0.; cosu = 1.; sinu = 0.; }
    const double aninv = sqrt(ax / mu);
    const double ecc_sq = sqrt(1. - ecc * ecc);
    double Pv[3], Qv[3];
    for (int k = 0; k < 3; k++) {
        Pv[k] = rinv * cosu * x[k] - aninv * sinu * v[k];
        Qv[k] = (rinv * sinu * x[k] + aninv * (cosu - ecc) * v[k]) / ecc_sq;
    }
    double l = u - ecc * sin(u);
    l += nn * dtime;
    u = solve_kepler(l, ecc);
    const double c2 = cos(u), s2 = sin(u);
    for (int k = 0; k < 3; k++) x[k] = ax * ((c2 - ecc) * Pv[k] + ecc_sq * s2 * Qv[k]);
    const double ri2 = sqrt(1. / dot3(x[0], x[1], x[2], x[0], x[1], x[2]));
    for (int k = 0; k < 3; k++) v[k] = ax * ax * nn * ri2 * (-s2 * Pv[k] + ecc_sq * c2 * Qv[k]);
}

__global__ void k_isolated(HP P, IsoView V, int n, double time_start, double time_end) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || V.number[i] != 0) return;
    double x[3], v[3], as[3], js[3], phs;
    ld3(V.pos, i, x);
    ld3(V.vel, i, v);
    const double zero[3] = {0., 0., 0.};
    if (eccentricity(P, x, v) < 0.8 && P.eps2_sun == 0.) {
        kepler_drift(P, x, v, time_end - time_start);
        V.time[i] += (time_end - time_start);
        st3(V.pos, i, x);
        st3(V.vel, i, v);
        V.phi_d[i] = 0.;
        st3(V.acc_d, i, zero);
        st3(V.jerk_d, i, zero);
        star_acc_jerk(P, x, v, as, js, &phs);
        st3(V.acc_s, i, as);
        st3(V.jerk_s, i, js);
        V.phi_s[i] = phs;
        V.dt[i] = dt_initial(P, V.time[i], V.dt[i], V.acc0[i], zero, zero, as, js);
    } else {
        // Sun-only Hermite in local time (FPHard: time_c = time, time = 0)
        const double time_c = V.time[i];
        double time = 0., dt = V.dt[i];
        star_acc_jerk(P, x, v, as, js, nullptr);
        double ad[3] = {0., 0., 0.}, jd[3] = {0., 0., 0.};
        ld3(V.acc_d, i, ad);
        ld3(V.jerk_d, i, jd);
        double a2s[3], a3s[3], a2d[3], a3d[3];
        for (long long it = 0; time < P.dt_tree && it < BLOCK_STEP_CAP; it++) {
            const double Dt = dt;
            double xp[3], vp[3], a0s[3], j0s[3], a0d[3], j0d[3];
            for (int k = 0; k < 3; k++) {
                a0s[k] = as[k]; j0s[k] = js[k]; a0d[k] = ad[k]; j0d[k] = jd[k];
                const double acc_sd = as[k] + ad[k], jerk_sd = js[k] + jd[k];
                xp[k] = x[k] + Dt * (v[k] + Dt * (SECONDORDER * acc_sd + THIRDORDER * Dt * jerk_sd));
                vp[k] = v[k] + Dt * (acc_sd + Dt * SECONDORDER * jerk_sd);
                ad[k] = 0.; jd[k] = 0.;
            }
            star_acc_jerk(P, xp, vp, as, js, nullptr);
            for (int ite = 0; ite < 2; ite++) {
                const double Dt2 = Dt * Dt, Dt_inv = recip_block(Dt), Dt_inv2 = Dt_inv * Dt_inv, Dt_inv3 = Dt_inv2 * Dt_inv;
                for (int k = 0; k < 3; k++) {
                    const double Am_s = as[k] - a0s[k], J0_s = Dt * j0s[k], J1_s = Dt * js[k];
                    const double A2_s = 3. * Am_s - (J1_s + 2. * J0_s), A3_s = -2. * Am_s + (J1_s + J0_s);
                    a2s[k] = 2. * Dt_inv2 * (A2_s + 3. * A3_s);
                    a3s[k] = 6. * Dt_inv3 * A3_s;
                    const double Am_d = ad[k] - a0d[k], J0_d = j0d[k] * Dt, J1_d = jd[k] * Dt;
                    const double A2_d = 3. * Am_d - (J1_d + 2. * J0_d), A3_d = -2. * Am_d + (J1_d + J0_d);
                    a2d[k] = 2. * (A2_d + 3. * A3_d) * Dt_inv2;
                    a3d[k] = 6. * A3_d * Dt_inv3;
                    const double A2_sd = A2_s + A2_d, A3_sd = A3_s + A3_d;
                    x[k] = xp[k] + ONE_SIXTIETH * Dt2 * (5. * A2_sd + 3. * ALPHA_POS * A3_sd);
                    v[k] = vp[k] + ONE_TWELFTH * Dt * (4. * A2_sd + 3. * A3_sd);
                }
                star_acc_jerk(P, x, v, as, js, nullptr);
            }
            time += dt;
            dt = dt_block(P, time, dt, V.acc0[i], ad, jd, a2d, a3d, as, js, a2s, a3s);
        }
        star_acc_jerk(P, x, v, as, js, &phs);
        st3(V.pos, i, x);
        st3(V.vel, i, v);
        st3(V.acc_s, i, as);
        st3(V.jerk_s, i, js);
        st3(V.acc_d, i, ad);
        st3(V.jerk_d, i, jd);
        V.phi_s[i] = phs;
        V.phi_d[i] = 0.;
        V.time[i] = time_c + time;
        V.dt[i] = dt;
    }
    V.n_cluster[i] = 1;
}

// ----------------------------------------------------------------- host

HP make_hp(const gplum_params &p) {
    HP h;
    h.m_sun = p.m_sun; h.eps2 = p.eps2; h.eps2_sun = p.eps2_sun; h.dt_tree = p.dt_tree;
    h.dt_min = p.dt_min; h.eta = p.eta; h.eta_0 = p.eta_0; h.eta_sun = p.eta_sun;
    h.eta_sun0 = p.eta_sun0; h.alpha2 = p.alpha2; h.cut = cutoff_of(p); h.collision = p.collision;
    h.terms_max = TERMS_MAX;
    return h;
}

static HardView hard_view(HardBuffers &hb) {
    HardView H{hb.pos.p, hb.vel.p, hb.acc_s.p, hb.jerk_s.p, hb.acc_d.p, hb.jerk_d.p, hb.xp.p, hb.vp.p,
               hb.a0_s.p, hb.j0_s.p, hb.a0_d.p, hb.j0_d.p, hb.a2_s.p, hb.a3_s.p, hb.a2_d.p, hb.a3_d.p,
               hb.mass.p, hb.rinv.p, hb.time.p, hb.dt.p, hb.acc0.p, hb.r_planet.p, hb.f.p, hb.phi_d.p,
               hb.phi_s.p, hb.id.p, hb.flags.p, hb.twin_of.p, hb.act.p};
    if (hb.crec_cap > 0) {
        H.crec = hb.crec.p;
        H.ccount = hb.ccount.p;
        H.ccap = hb.crec_cap;
    }
    return H;
}


// ------------------------------------------------------------ giant clusters
//
// Clusters above giant_min particles (the reference integrates clusters of 64 and more
// with OpenMP inside the cluster, hard.h:583-658) are spread over the whole GPU: each
// block step is a short sequence of kernels (predict all; collision test over all pairs
// with per-workgroup minima; decision and active flags; the active particles, one wave
// each, as on the global-memory path; the collision aftermath phase by phase; next
// block time and system time), launched in batches by the host, which checks a done
// flag between batches.  Same functions, same summation orders: results identical to the size-class
// kernels.
struct GiantState {
    double t_s, sys_time, ed;
    long long loop, pairs;
    int done, flag_col, ic, jc, n_col;
};

constexpr int GIANT_T = 256;          // threads per workgroup of the grid kernels
constexpr int GIANT_RED = 1024;       // threads of the one-workgroup kernels

__device__ inline void block_min2(double &u, double &v, double *s_u, double *s_v) {
    const int t = threadIdx.x;
    s_u[t] = u;
    s_v[t] = v;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (t < w) {
            if (s_u[t + w] < s_u[t]) s_u[t] = s_u[t + w];
            if (s_v[t + w] < s_v[t]) s_v[t] = s_v[t + w];
        }
        __syncthreads();
    }
    u = s_u[0];
    v = s_v[0];
    __syncthreads();
}

// initial calcGravity of all members with flags cleared (hermite.h:259-270)
__global__ __launch_bounds__(GIANT_T) void k_g_init(HP P, HardView H, int b, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gravity_full(P, H, b, n, i);
    H.flags[b + i] &= ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
    H.twin_of[b + i] = -1;
}

// loop state and the first block time: t_s = min(time + dt), sys_time = min(time) over
// the live members; done once sys_time reaches the end of the soft step or the cap
__global__ __launch_bounds__(GIANT_RED) void k_g_times(HP P, HardView H, int b, int n, GiantState *G, int first) {
    __shared__ double s_u[GIANT_RED], s_v[GIANT_RED];
    if (!first && G->done) return;
    double tl = 1.e10, tm = 1.e10;
    for (int i = threadIdx.x; i < n; i += blockDim.x)
        if (!(H.flags[b + i] & GPLUM_FLAG_DEAD)) {
            tl = dmin(tl, H.time[b + i] + H.dt[b + i]);
            tm = dmin(tm, H.time[b + i]);
        }
    block_min2(tl, tm, s_u, s_v);
    if (threadIdx.x != 0) return;
    if (first) {
        G->loop = 0;
        G->ed = 0.;
        G->n_col = 0;
        G->pairs = (long long)n * (long long)(n - 1);
        G->sys_time = 0.;
    } else {
        G->loop++;
        G->sys_time = tm;
    }
    G->t_s = tl;
    G->flag_col = 0;
    G->done = (G->sys_time < P.dt_tree && G->loop < BLOCK_STEP_CAP) ? 0 : 1;
}

__global__ __launch_bounds__(GIANT_T) void k_g_predict(HardView H, int b, int n, const GiantState *G) {
    if (G->done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    predict(H, b + i, G->t_s - H.time[b + i]);
}

// collisionDetermination over the pairs (i, j) of this workgroup: i from blockIdx.x,
// j from the chunk blockIdx.y; per-workgroup minimum in (R, i, j) order, which picks
// the pair the sequential search (ascending i, then j, strict <) finds
__device__ inline bool rij_less(double r, int i, int j, double r2, int i2, int j2) {
    return r < r2 || (r == r2 && (i < i2 || (i == i2 && j < j2)));
}

__global__ __launch_bounds__(GIANT_T) void k_g_collide(HardView H, int b, int n, const GiantState *G,
                                                       double *__restrict__ part_r, int *__restrict__ part_i,
                                                       int *__restrict__ part_j) {
    __shared__ double s_r[GIANT_T];
    __shared__ int s_i[GIANT_T], s_j[GIANT_T];
    if (G->done) return;
    const int t = threadIdx.x;
    const int i = blockIdx.x * blockDim.x + t;
    const int jchunk = (n + gridDim.y - 1) / gridDim.y;
    const int j0 = blockIdx.y * jchunk, j1 = min(n, j0 + jchunk);
    double rmin = 1.;
    int bi = 0x7fffffff, bj = 0x7fffffff;
    if (i < n && !(H.flags[b + i] & GPLUM_FLAG_DEAD)) {
        const double xi = H.xp[3 * (b + i)], yi = H.xp[3 * (b + i) + 1], zi = H.xp[3 * (b + i) + 2];
        const double fri = H.f[b + i] * H.r_planet[b + i];
        for (int j = j0; j < j1; j++) {
            if (i == j || (H.flags[b + j] & GPLUM_FLAG_DEAD)) continue;
            const double dx = xi - H.xp[3 * (b + j)];
            const double dy = yi - H.xp[3 * (b + j) + 1];
            const double dz = zi - H.xp[3 * (b + j) + 2];
            const double d2 = dot3(dx, dy, dz, dx, dy, dz);
            const double r2 = fri + H.f[b + j] * H.r_planet[b + j];
            if (!(d2 < COL_FILTER * r2 * r2)) continue;
            const double Rr = sqrt(d2) / r2;
            if (Rr < rmin) { rmin = Rr; bi = i; bj = j; }
        }
    }
    s_r[t] = rmin; s_i[t] = bi; s_j[t] = bj;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (t < w && rij_less(s_r[t + w], s_i[t + w], s_j[t + w], s_r[t], s_i[t], s_j[t])) {
            s_r[t] = s_r[t + w]; s_i[t] = s_i[t + w]; s_j[t] = s_j[t + w];
        }
        __syncthreads();
    }
    if (t == 0) {
        const int k = blockIdx.y * gridDim.x + blockIdx.x;
        part_r[k] = s_r[0]; part_i[k] = s_i[0]; part_j[k] = s_j[0];
    }
}

// the pair with the smallest R (< 1: a collision, the lighter body is the impactor; all
// live members are corrected to t_s), then the active flags of the step
__global__ __launch_bounds__(GIANT_RED) void k_g_decide(HP P, HardView H, int b, int n, GiantState *G,
                                                        const double *__restrict__ part_r,
                                                        const int *__restrict__ part_i,
                                                        const int *__restrict__ part_j, int nparts) {
    __shared__ double s_r[GIANT_RED];
    __shared__ int s_i[GIANT_RED], s_j[GIANT_RED];
    __shared__ int s_col;
    if (G->done) return;
    const int t = threadIdx.x;
    double r = 1.;
    int bi = 0x7fffffff, bj = 0x7fffffff;
    if (P.collision)
        for (int k = t; k < nparts; k += blockDim.x)
            if (rij_less(part_r[k], part_i[k], part_j[k], r, bi, bj)) { r = part_r[k]; bi = part_i[k]; bj = part_j[k]; }
    s_r[t] = r; s_i[t] = bi; s_j[t] = bj;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (t < w && rij_less(s_r[t + w], s_i[t + w], s_j[t + w], s_r[t], s_i[t], s_j[t])) {
            s_r[t] = s_r[t + w]; s_i[t] = s_i[t + w]; s_j[t] = s_j[t + w];
        }
        __syncthreads();
    }
    if (t == 0) {
        s_col = 0;
        if (s_r[0] < 1.) {
            const int gi = s_i[0], gj = s_j[0];
            s_col = 1;
            if (H.mass[b + gi] < H.mass[b + gj]) { G->ic = gi; G->jc = gj; } else { G->ic = gj; G->jc = gi; }
        }
        G->flag_col = s_col;
    }
    __syncthreads();
    const double t_s = G->t_s;
    const int col = s_col;
    for (int i = t; i < n; i += blockDim.x) {
        if (col) H.dt[b + i] = t_s - H.time[b + i];
        H.act[b + i] = !(H.flags[b + i] & GPLUM_FLAG_DEAD) && (col || H.time[b + i] + H.dt[b + i] == t_s);
    }
}

// the active members, one wave each (coop_correct_active over the whole grid)
__global__ __launch_bounds__(GIANT_T) void k_g_correct(HP P, HardView H, int b, int n, GiantState *G) {
    if (G->done) return;
    const JData J{H.xp + 3 * b, H.vp + 3 * b, H.mass + b, H.rinv + b, H.id + b};
    long long pairs = 0;
    const int waves = (int)(blockDim.x >> 6);
    coop_correct_active(P, H, J, b, n, G->t_s, G->flag_col, pairs, (int)blockIdx.x * waves + (int)(threadIdx.x >> 6),
                        (int)gridDim.x * waves);
    if ((threadIdx.x & 63) == 0 && pairs) atomicAdd((unsigned long long *)&G->pairs, (unsigned long long)pairs);
}

// perfect merging and its aftermath (the phases of collision_tail, each over the grid;
// all return at once in the block steps without a collision)
__global__ void k_g_merge(HP P, HardView H, int b, int n, GiantState *G) {
    if (G->done || !G->flag_col || threadIdx.x != 0) return;
    G->ed += perfect_merge(P, H, b, n, G->ic, G->jc);
    G->n_col++;
}
__global__ __launch_bounds__(GIANT_T) void k_g_tail_gravity(HP P, HardView H, int b, int n, GiantState *G) {
    if (G->done || !G->flag_col) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gravity_full(P, H, b, n, i);
    atomicAdd((unsigned long long *)&G->pairs, (unsigned long long)(n - 1));
}
__global__ __launch_bounds__(GIANT_T) void k_g_tail_merged(HardView H, int b, int n, const GiantState *G) {
    if (G->done || !G->flag_col) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (H.flags[b + i] & GPLUM_FLAG_MERGED)) merge_acc_jerk(H, b, n, i);
}
__global__ __launch_bounds__(GIANT_T) void k_g_tail_dt(HP P, HardView H, int b, int n, const GiantState *G) {
    if (G->done || !G->flag_col) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int g = b + i;
    if (!(H.flags[g] & GPLUM_FLAG_DEAD)) {
        double ad[3], jd[3], as[3], js[3];
        ld3(H.acc_d, g, ad); ld3(H.jerk_d, g, jd); ld3(H.acc_s, g, as); ld3(H.jerk_s, g, js);
        H.dt[g] = dt_initial(P, H.time[g], H.dt[g], H.acc0[g], ad, jd, as, js);
    }
}
__global__ __launch_bounds__(GIANT_T) void k_g_tail_twins(HardView H, int b, int n, const GiantState *G) {
    if (G->done || !G->flag_col) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && H.twin_of[b + i] >= 0) H.dt[b + i] = H.dt[b + H.twin_of[b + i]];
}

// final calcGravity with potentials (hermite.h:466-470), then the merged targets
__global__ __launch_bounds__(GIANT_T) void k_g_final(HP P, HardView H, int b, int n, GiantState *G) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gravity_full(P, H, b, n, i);
    atomicAdd((unsigned long long *)&G->pairs, (unsigned long long)(n - 1));
}
__global__ __launch_bounds__(GIANT_T) void k_g_final_merged(HardView H, int b, int n, const GiantState *G, int c,
                                                            double *edisp, int *ncol, long long *nblock,
                                                            long long *npair, double time_end) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && G->n_col > 0 && (H.flags[b + i] & GPLUM_FLAG_MERGED)) merge_acc_jerk(H, b, n, i);
    if (i == 0) {
        edisp[c] = G->ed;
        ncol[c] = G->n_col;
        nblock[c] = (G->sys_time < time_end) ? -1 : G->loop;
        npair[c] = G->pairs;
    }
}

// Giant clusters run concurrently, one per stream of a small per-device pool (streams
// at the default priority, created once and kept for the process).  Each slot captures
// GIANT_BATCH block steps of its cluster into a hipGraph once (10 kernels per step, no
// memset nodes; every kernel returns at once after the done flag is set) and replays it
// per round, then reads its done flag; a finished slot takes the next giant cluster.
// The graph keeps the host from spending its time on kernel launches.
constexpr int GIANT_BATCH = 32;
constexpr int GIANT_STREAMS = 8;

struct GiantSlot {
    int c = -1, b = 0, n = 0, g_n = 0, g_jc = 0, g_w = 0;
    GiantState *G = nullptr;
    double *r = nullptr;
    int *pi = nullptr, *pj = nullptr;
    hipGraphExec_t exec = nullptr;      // GIANT_BATCH block steps of this cluster
};

struct GiantPool {
    hipStream_t st[GIANT_STREAMS];
    hipEvent_t join[GIANT_STREAMS];
    hipEvent_t fork;
    int *done_h;          // pinned host copies of the slots' done flags (asynchronous reads)
};

// the calling thread's device's pool (created on first use)
static int giant_pool(GiantPool *out) {
    static std::mutex mu;
    static GiantPool pool[64] = {};
    int dev = 0;
    GPLUM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return fail(GPLUM_E_NODEVICE, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    GiantPool &p = pool[dev];
    for (int k = 0; k < GIANT_STREAMS; k++) {
        if (!p.st[k]) GPLUM_HIP(hipStreamCreateWithFlags(&p.st[k], hipStreamNonBlocking));
        if (!p.join[k]) GPLUM_HIP(hipEventCreateWithFlags(&p.join[k], hipEventDisableTiming));
    }
    if (!p.fork) GPLUM_HIP(hipEventCreateWithFlags(&p.fork, hipEventDisableTiming));
    if (!p.done_h) GPLUM_HIP(hipHostMalloc((void **)&p.done_h, sizeof(int) * GIANT_STREAMS, hipHostMallocDefault));
    *out = p;
    return GPLUM_OK;
}

static void giant_start(const HP &P, HardView &H, GiantSlot &g, hipStream_t st) {
    hipLaunchKernelGGL(k_g_init, dim3(g.g_n), dim3(GIANT_T), 0, st, P, H, g.b, g.n);
    hipLaunchKernelGGL(k_g_times, dim3(1), dim3(GIANT_RED), 0, st, P, H, g.b, g.n, g.G, 1);
}

static void giant_steps(const HP &P, HardView &H, GiantSlot &g, hipStream_t st) {
    for (int s = 0; s < GIANT_BATCH; s++) {
        hipLaunchKernelGGL(k_g_predict, dim3(g.g_n), dim3(GIANT_T), 0, st, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_collide, dim3(g.g_n, g.g_jc), dim3(GIANT_T), 0, st, H, g.b, g.n, g.G, g.r, g.pi, g.pj);
        hipLaunchKernelGGL(k_g_decide, dim3(1), dim3(GIANT_RED), 0, st, P, H, g.b, g.n, g.G, g.r, g.pi, g.pj,
                           g.g_n * g.g_jc);
        hipLaunchKernelGGL(k_g_correct, dim3(g.g_w), dim3(GIANT_T), 0, st, P, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_merge, dim3(1), dim3(64), 0, st, P, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_tail_gravity, dim3(g.g_n), dim3(GIANT_T), 0, st, P, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_tail_merged, dim3(g.g_n), dim3(GIANT_T), 0, st, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_tail_dt, dim3(g.g_n), dim3(GIANT_T), 0, st, P, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_tail_twins, dim3(g.g_n), dim3(GIANT_T), 0, st, H, g.b, g.n, g.G);
        hipLaunchKernelGGL(k_g_times, dim3(1), dim3(GIANT_RED), 0, st, P, H, g.b, g.n, g.G, 0);
    }
}

static void giant_finish(const HP &P, HardView &H, HardBuffers &hb, GiantSlot &g, hipStream_t st) {
    hipLaunchKernelGGL(k_g_final, dim3(g.g_n), dim3(GIANT_T), 0, st, P, H, g.b, g.n, g.G);
    hipLaunchKernelGGL(k_g_final_merged, dim3(g.g_n), dim3(GIANT_T), 0, st, H, g.b, g.n, g.G, g.c, hb.edisp.p,
                       hb.ncol.p, hb.nblock.p, hb.npair.p, P.dt_tree);
}

// Integrates the clusters listed in giants (host offsets off) on the giant path; the
// slots start after event fork (recorded on st once the cluster data were gathered) and
// st waits for all of them.
static int hard_giants(const HP &P, HardView &H, HardBuffers &hb, const std::vector<int> &giants,
                       const std::vector<int32_t> &off, hipStream_t st, const GiantPool &gp) {
    const hipStream_t *se = gp.st;
    int rc = GPLUM_OK;
    const int K = std::min<int>(GIANT_STREAMS, (int)giants.size());
    int max_n = 0;
    for (int c : giants) max_n = std::max(max_n, off[c + 1] - off[c]);
    const int max_parts = ceil_div(max_n, GIANT_T) * std::max(1, std::min(64, ceil_div(max_n, 64)));
    GPLUM_ENSURE(hb.g_state, sizeof(GiantState) * (size_t)K);
    GPLUM_ENSURE(hb.g_r, (size_t)max_parts * K);
    GPLUM_ENSURE(hb.g_i, (size_t)max_parts * K);
    GPLUM_ENSURE(hb.g_j, (size_t)max_parts * K);
    for (int k = 0; k < K; k++) GPLUM_HIP(hipStreamWaitEvent(se[k], gp.fork, 0));
    std::vector<GiantSlot> slot(K);
    size_t next = 0;
    auto release = [&](GiantSlot &g) {
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
        g.exec = nullptr;
    };
    auto assign = [&](int k) -> int {
        GiantSlot &g = slot[k];
        release(g);
        if (next >= giants.size()) { g.c = -1; return GPLUM_OK; }
        g.c = giants[next++];
        g.b = off[g.c];
        g.n = off[g.c + 1] - g.b;
        g.g_n = ceil_div(g.n, GIANT_T);
        g.g_jc = std::max(1, std::min(64, ceil_div(g.n, 64)));
        g.g_w = std::min(4096, ceil_div(g.n, GIANT_T / 64));
        g.G = reinterpret_cast<GiantState *>(hb.g_state.p) + k;
        g.r = hb.g_r.p + (size_t)k * max_parts;
        g.pi = hb.g_i.p + (size_t)k * max_parts;
        g.pj = hb.g_j.p + (size_t)k * max_parts;
        giant_start(P, H, g, se[k]);
        hipGraph_t graph = nullptr;
        GPLUM_HIP(hipStreamBeginCapture(se[k], hipStreamCaptureModeThreadLocal));
        giant_steps(P, H, g, se[k]);
        const hipError_t ec = hipStreamEndCapture(se[k], &graph);
        if (ec != hipSuccess) return fail(GPLUM_E_HIP, "graph capture of the giant-cluster steps failed");
        const hipError_t ei = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ei != hipSuccess) return fail(GPLUM_E_HIP, "graph instantiation of the giant-cluster steps failed");
        return GPLUM_OK;
    };
    for (int k = 0; k < K; k++)
        if ((rc = assign(k))) break;
    for (; !rc;) {
        bool any = false;
        for (int k = 0; k < K; k++)
            if (slot[k].c >= 0) {
                GPLUM_HIP(hipGraphLaunch(slot[k].exec, se[k]));
                GPLUM_HIP(hipMemcpyAsync(&gp.done_h[k], &slot[k].G->done, sizeof(int), hipMemcpyDeviceToHost,
                                         se[k]));
                any = true;
            }
        if (!any) break;
        GPLUM_HIP(hipGetLastError());
        for (int k = 0; k < K; k++)
            if (slot[k].c >= 0) {
                GPLUM_HIP(hipStreamSynchronize(se[k]));
                if (gp.done_h[k]) {
                    giant_finish(P, H, hb, slot[k], se[k]);
                    if ((rc = assign(k))) break;
                }
            }
    }
    for (int k = 0; k < K; k++) release(slot[k]);
    if (rc) return rc;
    // st waits for every slot
    for (int k = 0; k < K; k++) {
        GPLUM_HIP(hipEventRecord(gp.join[k], se[k]));
        GPLUM_HIP(hipStreamWaitEvent(st, gp.join[k], 0));
    }
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

// The size classes of the batched launch and their kernels; each class has a queue counter
// of its own.  A class of T threads evaluates T / n bodies' pair terms per round, and most
// block steps correct fewer bodies than that.  The lines (us per block step of one cluster):
// 16 members on one wave 5.9-7.2, on 256 threads 5.2-5.4, but four clusters per CU instead of
// one or two, which decides for batches; 32 on 256 threads 6.1-7.4, on 128 6.7-9.6; 64 on 512
// threads 8.8-9.4, on 256 10.2-10.9.
static int class_hi(int cls, int lds_max) {
    return cls == 0 ? HERMITE_SMALL : cls == 1 ? HERMITE_MID : cls == 2 ? HARD_SEQ_MAX : cls == 3 ? lds_max : 0x7fffffff;
}
static int class_lo(int cls, int lds_max) { return cls == 0 ? 0 : class_hi(cls - 1, lds_max); }
static void launch_class(int cls, bool dyadic, const HP &P, const HardView &H, const ClusterArgs &A, int grid, int lo, int hi,
                         hipStream_t st) {
    switch (cls) {
    case 0:
        if (dyadic) hipLaunchKernelGGL(k_hermite_small<true>, dim3(grid), dim3(HERMITE_BLOCK), 0, st, P, H, A, lo, hi);
        else hipLaunchKernelGGL(k_hermite_small<false>, dim3(grid), dim3(HERMITE_BLOCK), 0, st, P, H, A, lo, hi);
        break;
    case 1: hipLaunchKernelGGL((k_hermite_mid<HERMITE_SMALL + 1, HERMITE_MID, 256>), dim3(grid), dim3(256), 0, st, P, H, A, lo, hi); break;
    case 2: hipLaunchKernelGGL((k_hermite_mid<HERMITE_MID + 1, HARD_SEQ_MAX, 512>), dim3(grid), dim3(512), 0, st, P, H, A, lo, hi); break;
    case 3: hipLaunchKernelGGL(k_hermite_big, dim3(grid), dim3(HERMITE_BIG_BLOCK), 0, st, P, H, A, lo, hi); break;
    default:
        hipLaunchKernelGGL(k_hermite_global, dim3(grid), dim3(HERMITE_GLOBAL_BLOCK), 0, st, P, H, A, lo, hi);
    }
}

// zeroes the cluster-queue counters (a kernel, not a memset, so that the launch
// sequence can be captured into a graph and replayed)
__global__ void k_reset_queue(int *next) {
    if (threadIdx.x < HERMITE_QUEUES) next[threadIdx.x] = 0;
}

int hard_launch(const gplum_params &p, HardBuffers &hb, int ncl, const int32_t *d_off,
                const int32_t *d_order, bool persistent, int n_cu, hipStream_t st, HardStreams &hs,
                int wg_per_cu, int lds_max, int giant_min, int terms_max, int n_off_grid) {
    if (ncl <= 0) return GPLUM_OK;
    HP P = make_hp(p);
    P.terms_max = std::max(0, std::min(TERMS_MAX, terms_max));
    const bool dyadic = dyadic_tree(p) && n_off_grid < ncl;   // every cluster off the grid: on st itself
    HardView H = hard_view(hb);
    GPLUM_ENSURE(hb.next, HERMITE_QUEUES);
    GPLUM_ENSURE(hb.edisp, ncl);
    GPLUM_ENSURE(hb.ncol, ncl);
    GPLUM_ENSURE(hb.nblock, ncl);
    GPLUM_ENSURE(hb.npair, ncl);
    hipLaunchKernelGGL(k_reset_queue, dim3(1), dim3(64), 0, st, hb.next.p);
    lds_max = std::min(HERMITE_LDS, std::max(HARD_SEQ_MAX, lds_max));
    const int grid = persistent ? std::min(ncl, std::max(1, n_cu) * std::max(1, wg_per_cu)) : ncl;
    const bool big = hb.max_size > HERMITE_SMALL;
    if (!dyadic) n_off_grid = 0;
    if (big || n_off_grid > 0) {
        int rc = hs.ensure();
        if (rc) return rc;
        GPLUM_HIP(hipEventRecord(hs.fork, st));
    }
    giant_min = std::max(HARD_SEQ_MAX, giant_min);
    // giant clusters start right after the gather: their stream pool waits on this event
    GiantPool gpool{};
    if (hb.max_size > giant_min) {
        int rc = giant_pool(&gpool);
        if (rc) return rc;
        GPLUM_HIP(hipEventRecord(gpool.fork, st));
    }
    ClusterArgs A{d_off, d_order, ncl, persistent ? 1 : 0, hb.next.p, hb.edisp.p, hb.ncol.p, hb.nblock.p, hb.npair.p};
    bool launched[HERMITE_CLASSES] = {};
    for (int k = 0; k < HERMITE_CLASSES; k++) {
        const int cls = HERMITE_CLASSES - 1 - k;               // the longest chains first
        const int lo = class_lo(cls, lds_max), hi = std::min(class_hi(cls, lds_max), giant_min);
        if (cls > 0 && (hb.max_size <= lo || hi <= lo)) continue;
        A.next = hb.next.p + cls;
        A.ncl = (cls == 0) ? ncl - n_off_grid : ncl;
        if (A.ncl <= 0) continue;
        if (cls > 0) GPLUM_HIP(hipStreamWaitEvent(hs.s[cls - 1], hs.fork, 0));
        launch_class(cls, dyadic, P, H, A, grid, lo, hi, cls > 0 ? hs.s[cls - 1] : st);
        if (cls > 0) GPLUM_HIP(hipEventRecord(hs.join[cls - 1], hs.s[cls - 1]));
        launched[cls] = true;
    }
    if (n_off_grid > 0) {
        // on a stream and a queue of their own, beside the other clusters
        hipStream_t so = hs.s[HERMITE_CLASSES - 1];
        ClusterArgs O = A;
        O.order = d_order + (ncl - n_off_grid);
        O.ncl = n_off_grid;
        O.next = hb.next.p + HERMITE_CLASSES;
        GPLUM_HIP(hipStreamWaitEvent(so, hs.fork, 0));
        launch_class(0, false, P, H, O, std::min(grid, n_off_grid), 0, HERMITE_SMALL, so);
        GPLUM_HIP(hipEventRecord(hs.join[HERMITE_CLASSES - 1], so));
    }
    if (hb.max_size > giant_min) {
        // giant clusters: several at a time over the whole GPU on a stream pool (the
        // size-class kernels above run meanwhile)
        std::vector<int32_t> off(ncl + 1);
        GPLUM_HIP(hipMemcpyAsync(off.data(), d_off, sizeof(int32_t) * (ncl + 1), hipMemcpyDeviceToHost, st));
        GPLUM_HIP(hipStreamSynchronize(st));
        std::vector<int> giants;
        for (int c = 0; c < ncl; c++)
            if (off[c + 1] - off[c] > giant_min) giants.push_back(c);
        // largest first
        std::stable_sort(giants.begin(), giants.end(),
                         [&](int x, int y) { return off[x + 1] - off[x] > off[y + 1] - off[y]; });
        int rc = hard_giants(P, H, hb, giants, off, st, gpool);
        if (rc) return rc;
    }
    for (int cls = 1; cls < HERMITE_CLASSES; cls++)
        if (launched[cls]) GPLUM_HIP(hipStreamWaitEvent(st, hs.join[cls - 1], 0));
    if (n_off_grid > 0) GPLUM_HIP(hipStreamWaitEvent(st, hs.join[HERMITE_CLASSES - 1], 0));
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

// Sun + hard acc/jerk at the current state and the first block step
// (calcGravity + calcDeltatInitial, gravity_hard.h:203-256, particle.h:886-914) of
// every particle of clusters [d_off[c], d_off[c+1]): one 64-thread block per cluster.
__global__ __launch_bounds__(HERMITE_BLOCK) void k_hard_prepare(HP P, HardView H, const int32_t *__restrict__ d_off,
                                                                int ncl) {
    const int c = blockIdx.x;
    if (c >= ncl) return;
    const int b = d_off[c], n = d_off[c + 1] - b;
    for (int i = (int)threadIdx.x; i < n; i += HERMITE_BLOCK) {
        gravity_full(P, H, b, n, i);
        double ad[3], jd[3], as[3], js[3];
        ld3(H.acc_d, b + i, ad); ld3(H.jerk_d, b + i, jd);
        ld3(H.acc_s, b + i, as); ld3(H.jerk_s, b + i, js);
        H.dt[b + i] = dt_initial(P, H.time[b + i], H.dt[b + i], H.acc0[b + i], ad, jd, as, js);
    }
}

int hard_prepare(const gplum_params &p, HardBuffers &hb, int ncl, const int32_t *d_off, hipStream_t st) {
    if (ncl <= 0) return GPLUM_OK;
    HP P = make_hp(p);
    HardView H{hb.pos.p, hb.vel.p, hb.acc_s.p, hb.jerk_s.p, hb.acc_d.p, hb.jerk_d.p, hb.xp.p, hb.vp.p,
               hb.a0_s.p, hb.j0_s.p, hb.a0_d.p, hb.j0_d.p, hb.a2_s.p, hb.a3_s.p, hb.a2_d.p, hb.a3_d.p,
               hb.mass.p, hb.rinv.p, hb.time.p, hb.dt.p, hb.acc0.p, hb.r_planet.p, hb.f.p, hb.phi_d.p,
               hb.phi_s.p, hb.id.p, hb.flags.p, hb.twin_of.p, hb.act.p};
    hipLaunchKernelGGL(k_hard_prepare, dim3(ncl), dim3(HERMITE_BLOCK), 0, st, P, H, d_off, ncl);
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

int hard_launch_single(const gplum_params &p, HardBuffers &hb, int c, int n_c, const int32_t *d_off,
                       hipStream_t st, bool off_grid) {
    // one launch integrating cluster c (n_c particles) only: the per-cluster-launch comparator
    HP P = make_hp(p);
    HardView H = hard_view(hb);
    const ClusterArgs A{d_off + c, nullptr, 1, 0, hb.next.p, hb.edisp.p + c, hb.ncol.p + c, hb.nblock.p + c, hb.npair.p + c};
    int cls = 0;
    while (n_c > class_hi(cls, HERMITE_LDS)) cls++;
    launch_class(cls, dyadic_tree(p) && !off_grid, P, H, A, 1, 0, 0x7fffffff, st);
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

int isolated_launch(const gplum_params &p, const IsoArgs &a, int n, double t0, double t1, hipStream_t st) {
    if (n <= 0) return GPLUM_OK;
    HP P = make_hp(p);
    IsoView V{a.pos, a.vel, a.acc_d, a.jerk_d, a.acc_s, a.jerk_s, a.phi_d, a.phi_s, a.time, a.dt, a.acc0,
              a.number, a.n_cluster};
    hipLaunchKernelGGL(k_isolated, dim3(ceil_div(n, 128)), dim3(128), 0, st, P, V, n, t0, t1);
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}


// ------------------------------------------------------- time-step self-check

__device__ inline uint64_t mix64(uint64_t z) {     // splitmix64 finaliser
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
// sign * [0.5, 1) * 2^e with e uniform in [e0, e1]
__device__ inline double rnd_mag(uint64_t &st, int e0, int e1) {
    st += 0x9E3779B97F4A7C15ULL;
    const uint64_t r = mix64(st);
    const double m = 0.5 + 0.5 * (double)(r >> 11) * 0x1p-53;
    const int e = e0 + (int)(mix64(r ^ 0x5851F42D4C957F2DULL) % (uint64_t)(e1 - e0 + 1));
    return ((r >> 10) & 1) ? -ldexp(m, e) : ldexp(m, e);
}

// A random state: accelerations and their derivatives over many decades (wide: every magnitude
// spread by another 2^+-wide), a step dt_tree 2^-kk, kk <= k_max, and a time on the step's grid.
struct DtSample {
    double v[8][3], acc0, dt, time;      // v: acc, jerk, snap, crackle of the planets, of the Sun
};
__device__ inline void dt_sample(const HP &P, uint64_t &st, int wide, int k_max, DtSample &s) {
    const int e_lo[8] = {-20, -24, -28, -32, -12, -16, -20, -24};
    const int e_hi[8] = {8, 14, 20, 26, 4, 8, 12, 16};
    for (int q = 0; q < 8; q++)
        for (int k = 0; k < 3; k++) s.v[q][k] = rnd_mag(st, e_lo[q] - wide, e_hi[q] + wide);
    s.acc0 = fabs(rnd_mag(st, -12, 4));
    st += 0x9E3779B97F4A7C15ULL;
    const uint64_t r = mix64(st);
    const int kk = 1 + (int)(r % (uint64_t)k_max);
    s.dt = ldexp(P.dt_tree, -kk);
    s.time = s.dt * (double)((r >> 8) % (1ULL << kk));
}
template <bool FAST>
__device__ inline double dt_of(const HP &P, const DtSample &s, int *fell = nullptr) {
    return dt_block<FAST>(P, s.time + s.dt, s.dt, s.acc0, s.v[0], s.v[1], s.v[2], s.v[3], s.v[4], s.v[5], s.v[6], s.v[7], fell);
}

// dt_block with the fast criterion against dt_block with calc_dt4 on random states.  One sample
// in four is spread by 2^+-540, so that the products of squares in the fast criterion underflow
// below DBL_MIN or overflow past DBL_MAX.  Counts results that differ in any bit and fast values
// sent to the exact evaluation.
__global__ void k_dt_selfcheck(HP P, long long n, uint64_t seed, unsigned long long *out) {
    unsigned long long mism = 0, fb = 0;
    for (long long s = blockIdx.x * (long long)blockDim.x + threadIdx.x; s < n; s += (long long)gridDim.x * blockDim.x) {
        uint64_t st = seed ^ mix64((uint64_t)s * 0x2545F4914F6CDD1DULL);
        DtSample d;
        dt_sample(P, st, ((s & 3) == 3) ? 540 : 0, 30, d);
        int fell = 0;
        const double a = dt_of<true>(P, d, &fell), b = dt_of<false>(P, d);
        mism += (__double_as_longlong(a) != __double_as_longlong(b)) ? 1 : 0;
        fb += fell;
    }
    atomicAdd(&out[0], mism);
    atomicAdd(&out[1], fb);
}

// The helpers of the lane-per-term and LDS paths, which act on a whole wave, one wave per sample:
//   roots      8 values per lane through root_and_inverse and inverse_and_root against sqrt and 1 / x.
//              One lane that a helper has to send to the library takes its whole wave there, so such
//              values (out of range; a low word of ones) come in one wave of eight each and the others
//              hold none: random mantissas, those next to a power of two or to a square, where a
//              rounding is closest.  Counts the values whose wave kept to the estimate.
//   steps      dt_block_rows of 2, 3 and 4 bodies (the sample number picks) on both kinds of grid and
//              dt_block_quad, a state per particle in the lanes of its quads, against dt_block with
//              calc_dt4.  Of eight samples one is wide (see dt_sample), three have derivatives scaled to
//              dt_1 = dt 2^k (1 + d), |d| from 2^-8 to 2^-51 or 0, around the 2^-10 margin and the grid
//              itself, and one has dt 3/4 of a power of two (not through the dyadic rule).
enum { CHK_ROOTS, CHK_ROOTS_FAST, CHK_ROOTS_BAD, CHK_STEPS, CHK_STEPS_NEAR, CHK_ROWS_BAD, CHK_DYADIC, CHK_DYADIC_BAD, CHK_QUAD_BAD,
       CHK_N };
__device__ inline bool bits_differ(double a, double b) { return __double_as_longlong(a) != __double_as_longlong(b); }

template <int N>
__device__ inline void check_rows(const HP &P, bool dyadic_p, int k_max, long long q, uint64_t seed, int mode,
                                  unsigned long long cnt[CHK_N]) {
    const int L = (int)threadIdx.x;
    const int T = (N == 2) ? ((L >> 4) & 1) : (L >> 4), p = (N == 2) ? ((L >> 2) & 1) : ((L >> 2) & 3), c = L & 3;
    const bool sun = T == 0, pad = c == 3;
    uint64_t st = seed ^ mix64((uint64_t)(q * 4 + p) * 0x2545F4914F6CDD1DULL);
    DtSample d;
    dt_sample(P, st, mode == 3 ? 540 : 0, k_max, d);
    const bool off_grid = mode == 2, near = mode >= 5;
    if (off_grid) {
        d.dt *= 0.75;
        d.time = 0.75 * d.time;
    }
    if (near) {
        const double dt_1 = dmin(calc_dt4(P.eta, P.alpha2, d.acc0, d.v[0], d.v[1], d.v[2], d.v[3]),
                                 calc_dt4(P.eta_sun, P.alpha2, 0., d.v[4], d.v[5], d.v[6], d.v[7]));
        st += 0x9E3779B97F4A7C15ULL;
        const uint64_t r = mix64(st);
        const int e = 8 + (int)((r >> 4) % 45);
        const double delta = (e == 52) ? 0. : ((r & 1) ? 1. : -1.) * ldexp(1., -e);
        const double lam = dt_1 / (ldexp(d.dt, (int)((r >> 1) & 3) - 2) * (1. + delta));
        for (int k = 0; k < 3; k++)
            for (int b = 0; b < 8; b += 4) {
                d.v[b + 1][k] *= lam;
                d.v[b + 2][k] *= lam * lam;
                d.v[b + 3][k] *= lam * lam * lam;
            }
    }
    const double want = dt_of<false>(P, d);
    double z[8];
    for (int b = 0; b < 8; b++) z[b] = pad ? 0. : (c == 0 ? d.v[b][0] : c == 1 ? d.v[b][1] : d.v[b][2]);
    const TermConsts C(P);
    const double za = sun ? z[4] : z[0], zj = sun ? z[5] : z[1], zs = sun ? z[6] : z[2], zc = sun ? z[7] : z[3];
    const double eta = sun ? P.eta_sun : P.eta, acc0 = sun ? 0. : d.acc0;
    cnt[CHK_STEPS]++;
    cnt[CHK_STEPS_NEAR] += near;
    cnt[CHK_ROWS_BAD] += bits_differ(dt_block_rows<N, false>(C, d.time + d.dt, d.dt, eta, acc0, za, zj, zs, zc), want);
    if (dyadic_p && !off_grid) {
        cnt[CHK_DYADIC]++;
        cnt[CHK_DYADIC_BAD] += bits_differ(dt_block_rows<N, true>(C, d.time + d.dt, d.dt, eta, acc0, za, zj, zs, zc), want);
    }
    cnt[CHK_QUAD_BAD] += bits_differ(dt_block_quad(P, d.time + d.dt, d.dt, d.acc0, z[0], z[1], z[2], z[3], z[4], z[5], z[6], z[7]),
                                     want);
}

__global__ __launch_bounds__(64) void k_path_selfcheck(HP P, bool dyadic_p, int k_max, long long n, uint64_t seed,
                                                       unsigned long long *out) {
    unsigned long long cnt[CHK_N] = {};
    for (long long q = blockIdx.x; q < n; q += gridDim.x) {
        const int mode = (int)(q & 7);
        uint64_t st = ~seed ^ mix64((uint64_t)(q * 64 + (int)threadIdx.x) * 0x2545F4914F6CDD1DULL);
        for (int v = 0; v < 8; v++) {
            double x = fabs(rnd_mag(st, -398, 398));
            st += 0x9E3779B97F4A7C15ULL;
            // (just below a power of two, value or root have a low word of ones)
            const uint64_t u = mix64(st), ulps = (u >> 58) + ((mode < 6 && !(u & 4)) ? 4 : 0);
            if ((u & 3) == 1) x = ldexp(1.0, (int)(u >> 8 & 511) - 256) * (1.0 + ((u & 4) ? 1. : -0.5) * 0x1p-52 * (double)ulps);
            if ((u & 3) == 2) {
                const double w = fabs(rnd_mag(st, -198, 198));
                x = __longlong_as_double(__double_as_longlong(w * w) + (long long)ulps - 32);
            }
            if (mode == 6 && (u & 48) == 0) x = __longlong_as_double(__double_as_longlong(x) | 0xFFFFFFFFll);
            if (mode == 7 && (u & 48) == 0) x = fabs(rnd_mag(st, -1000, 1000));
            double rt, rtinv, sinv, root;
            root_and_inverse(x, true, rt, rtinv);
            inverse_and_root(x, sinv, root);
            const double r0 = sqrt(x), s0 = 1. / x;
            const bool library = __ballot(!root_range(x) || rcp_exception(x) || rcp_exception(r0)) != 0;
            cnt[CHK_ROOTS]++;
            cnt[CHK_ROOTS_FAST] += !library;
            cnt[CHK_ROOTS_BAD] += bits_differ(rt, r0) || bits_differ(rtinv, 1. / r0) || bits_differ(sinv, s0) ||
                                  bits_differ(root, sqrt(s0));
        }
        const int bodies = 2 + (int)((q >> 3) % 3);
        if (bodies == 2) check_rows<2>(P, dyadic_p, k_max, q, seed, mode, cnt);
        else if (bodies == 3) check_rows<3>(P, dyadic_p, k_max, q, seed, mode, cnt);
        else check_rows<4>(P, dyadic_p, k_max, q, seed, mode, cnt);
    }
    for (int k = 0; k < CHK_N; k++)
        if (cnt[k]) atomicAdd(&out[k], cnt[k]);
}

int hermite_path_selfcheck(const gplum_params &p, long long n, uint64_t seed, int64_t counts[CHK_N]) {
    if (n < 0) return fail(GPLUM_E_ARG, "negative sample count");
    if (!(p.dt_tree > 0.) || !(p.dt_min > 0.) || p.dt_min > 0.25 * p.dt_tree)
        return fail(GPLUM_E_ARG, "dt_min must lie in (0, dt_tree / 4]");
    DArray<unsigned long long> cnt;
    GPLUM_ENSURE(cnt, CHK_N);
    GPLUM_HIP(hipMemset(cnt.p, 0, CHK_N * sizeof(unsigned long long)));
    // no sample's step lies below dt_min, as the dyadic rule asks
    int k_max = 1;
    while (k_max < 30 && std::ldexp(p.dt_tree, -(k_max + 1)) >= p.dt_min) k_max++;
    hipLaunchKernelGGL(k_path_selfcheck, dim3(1024), dim3(64), 0, 0, make_hp(p), dyadic_tree(p), k_max, n, seed, cnt.p);
    GPLUM_HIP(hipGetLastError());
    unsigned long long h[CHK_N] = {};
    GPLUM_HIP(hipMemcpy(h, cnt.p, sizeof(h), hipMemcpyDeviceToHost));
    for (int k = 0; k < CHK_N; k++) counts[k] = (int64_t)h[k];
    return GPLUM_OK;
}

int hermite_dt_selfcheck(const gplum_params &p, long long n, uint64_t seed, long long *mismatches,
                         long long *fallbacks) {
    if (n < 0) return fail(GPLUM_E_ARG, "negative sample count");
    DArray<unsigned long long> cnt;
    GPLUM_ENSURE(cnt, 2);
    GPLUM_HIP(hipMemset(cnt.p, 0, 2 * sizeof(unsigned long long)));
    hipLaunchKernelGGL(k_dt_selfcheck, dim3(1024), dim3(256), 0, 0, make_hp(p), n, seed, cnt.p);
    GPLUM_HIP(hipGetLastError());
    unsigned long long h[2] = {0, 0};
    GPLUM_HIP(hipMemcpy(h, cnt.p, sizeof(h), hipMemcpyDeviceToHost));
    if (mismatches) *mismatches = (long long)h[0];
    if (fallbacks) *fallbacks = (long long)h[1];
    return GPLUM_OK;
}

}  // namespace gplum
