// hermite_lds.hpp -- block steps of one cluster by one workgroup with the whole cluster
// in LDS (included by hermite.hip, whose pair, Sun, time-step and quad helpers it uses).
//
// A block step corrects few of a cluster's particles (2 to 7 on average for clusters of 5
// to 256), but each of them needs its force from every member three times, one after the
// other: the step's length is the latency of that chain.  The work of one force evaluation
// is therefore spread over the whole workgroup, in two phases between barriers:
//   terms       one (body, partner) pair per thread, T / n bodies at a time; the Sun's terms
//               by the quads meanwhile;
//   quads       four lanes per body (x, y, z and a padding lane): the pair terms added in
//               ascending j (clusters up to HARD_SEQ_MAX; larger ones add theirs as the
//               64-partial butterfly on eight lanes per component, in a phase of its own),
//               mergeAccJerk for merged bodies, corrector.
// A merged target's twins are bodies of their own, so a family costs no more than as many
// active particles.  Same operations in the same order as the reference's loops
// (hermite.h:224-479), so the results are those of the other paths bit for bit.
//
// What bounds it: the latency of three evaluations, one after the other: waves wait 56 to 72 % of
// their cycles.  64 members, 3.4 bodies corrected, 18,000 cycles per block step: pair terms (each a
// correctly rounded FP64 square root and reciprocal, and the loads before it) 2,600, 1,800 and 1,800,
// sums over j with corrections, step choice and stores 3,100, 2,400 and 3,900, prediction, lists and
// next time 2,300; 128 members, 22,000: evaluations 4,600, 4,300 and 4,300 with their sums.  The
// chip's FP64 rate is far away (a cluster occupies one CU).  Measured on one cluster, us per
// block step, against one lane per particle in registers and, from the first merger on, one
// lane per particle in global memory (up to 64 members), or lane groups of 8 to 64 lanes (above):
// 8 members 5.6 -> 4.9, 16 20 -> 6.0, 32 44 -> 6.1 (2 to 4 bodies corrected, one merger), 64 152
// -> 8.8, 96 23 -> 10.6, 128 23 -> 11.1, 256 99 -> 33 (18 bodies, 61 mergers).
#pragma once

namespace gplum {

template <int NMAX>
struct ClusterLds {
    double pos[3 * NMAX], vel[3 * NMAX], acc_s[3 * NMAX], jerk_s[3 * NMAX], acc_d[3 * NMAX], jerk_d[3 * NMAX];
    double xp[3 * NMAX], vp[3 * NMAX];         // predicted: the partners' state of a block step
    double bx[3 * NMAX], bv[3 * NMAX];         // corrected state of the bodies (by slot)
    double fa[6 * NMAX];                       // hard force of the bodies (by slot): families, waves' sums
    double mass[NMAX], rinv[NMAX], time[NMAX], dt[NMAX], acc0[NMAX], r_planet[NMAX], f[NMAX];
    double fr[NMAX];                           // f r_planet of the live members, NaN of the dead
    int64_t id[NMAX];
    int32_t flags[NMAX], twin_of[NMAX];
    int32_t first[NMAX], next[NMAX];           // a target's twins, ascending (-1 ends the list)
    int32_t body[NMAX], slot_of[NMAX];         // the bodies of a block step, ascending
    int32_t nb, anym;                          // their number, any merged one
    int32_t hit;                               // a pair may collide
    double red_r[16];
    int32_t red_lo[16], red_hi[16];
};

// star_acc_jerk of a quad's particle, one component per lane (see quad_sum).
__device__ inline void star_quad(const HP &P, double x, double v, bool pad, double &as, double &js) {
    const double dr = -x, dv = -v;
    double r2inv, rinv;
    inverse_and_root(quad_sq(dr) + P.eps2_sun, r2inv, rinv);
    const double r3inv = rinv * r2inv;
    const double mj = P.m_sun * r3inv;
    const double alpha = quad_dot(dr, dv, pad) * r2inv;
    as = mj * dr;
    js = mj * (dv - 3. * alpha * dr);
}

// dt_block of a quad's particle, one component per lane.
__device__ inline double dt_block_quad(const HP &P, double time, double dt, double acc0, double ad, double jd,
                                       double a2d, double a3d, double as, double js, double a2s, double a3s) {
    bool cap;
    const double dt_0 = dt_candidate(time, dmin(2. * dt, 0.5 * P.dt_tree), cap);
    const double f_planet = dt4_fast_quad(P.eta, P.alpha2, acc0, ad, jd, a2d, a3d);
    const double f_sun = dt4_fast_quad(P.eta_sun, P.alpha2, 0., as, js, a2s, a3s);
    double dt_1 = dmin(f_planet, f_sun);
    if (!(f_planet <= DBL_MAX && f_sun <= DBL_MAX) || !clear_of_steps(dt_1, dt_0))
        dt_1 = dmin(dt4_quad(P.eta, P.alpha2, acc0, ad, jd, a2d, a3d),
                    dt4_quad(P.eta_sun, P.alpha2, 0., as, js, a2s, a3s));
    const double dt_next = dt_reduce(dt_0, dt_1, dt);
    return (cap || dt_next < 2. * P.dt_min) ? P.dt_min : dt_next;
}

// The smallest f(time, dt) of the live members, in every lane (every lane of a wave calls it).
template <int NMAX, class F>
__device__ inline double lds_min(const ClusterLds<NMAX> &C, int n, F f) {
    double m = 1.e10;
    for (int i0 = 0; i0 < n; i0 += 64) {
        const int i = min(i0 + (int)(threadIdx.x & 63), n - 1);   // the last member again: no harm to a minimum
        const double v = f(C.time[i], C.dt[i]);
        m = __builtin_fmin(m, (C.flags[i] & GPLUM_FLAG_DEAD) ? 1.e10 : v);
    }
    m = row_min(m);
    double r = readlane_f64(m, 0);
#pragma unroll
    for (int l = 16; l < min(NMAX, 64); l += 16) r = __builtin_fmin(r, readlane_f64(m, l));
    return r;
}
// the next block time
template <int NMAX>
__device__ inline double lds_next_time(const ClusterLds<NMAX> &C, int n) {
    return lds_min(C, n, [](double time, double dt) { return time + dt; });
}
// The system time, as far as the loop asks: the smallest time of the live members once the
// next block time t_s has reached time_end; before that some member's time, and so the
// system's, is below t_s.
template <int NMAX>
__device__ inline double lds_system_time(const ClusterLds<NMAX> &C, int n, double t_s, double time_end, double before) {
    if (t_s < time_end) return before;
    return lds_min(C, n, [](double time, double) { return time; });
}

// The bodies of a block step, by one wave: the active members (all live ones after a
// collision) and the twins of the merged ones among them.
template <int NMAX>
__device__ inline void lds_bodies(ClusterLds<NMAX> &C, int n, double t_s, bool col) {
    constexpr int NW = (NMAX + 63) / 64;
    const int lane = (int)(threadIdx.x & 63);
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long act[NW], merged = 0ull;
#pragma unroll
    for (int u = 0; u < NW; u++) {
        const int i = 64 * u + lane;
        bool a = false, m = false;
        if (i < n) {
            const int fl = C.flags[i];
            a = !(fl & GPLUM_FLAG_DEAD) && (col || C.time[i] + C.dt[i] == t_s);
            m = a && (fl & GPLUM_FLAG_MERGED);
        }
        act[u] = __ballot(a);
        merged |= __ballot(m);
    }
    int base = 0;
#pragma unroll
    for (int u = 0; u < NW; u++) {
        const int i = 64 * u + lane;
        bool b = (act[u] >> lane) & 1ull;
        if (merged && i < n) {
            const int tg = C.twin_of[i];
            if (tg >= 0) {
#pragma unroll
                for (int q = 0; q < NW; q++) b = b || ((tg >> 6) == q && ((act[q] >> (tg & 63)) & 1ull));
            }
        }
        const unsigned long long mb = __ballot(b);
        if (b) {
            const int s = base + __popcll(mb & below);
            C.body[s] = i;
            C.slot_of[i] = s;
        }
        base += __popcll(mb);
    }
    if (lane == 0) {
        C.nb = base;
        C.anym = merged != 0ull;
    }
}

// f r_planet and the twin lists, after loading and after a merger
template <int NMAX, int T>
__device__ inline void lds_relations(ClusterLds<NMAX> &C, int n) {
    for (int i = (int)threadIdx.x; i < n; i += T) {
        C.fr[i] = (C.flags[i] & GPLUM_FLAG_DEAD) ? __builtin_nan("") : C.f[i] * C.r_planet[i];
        const int tw = C.twin_of[i];
        int first = -1, next = -1;
        for (int j = n - 1; j >= 0; j--) {
            const int tj = C.twin_of[j];
            if (tj == i) first = j;
            if (j > i && tw >= 0 && tj == tw) next = j;
        }
        C.first[i] = first;
        C.next[i] = next;
    }
}

// Sun and hard acc/jerk of every member at its current state, one thread each
template <int NMAX, int T>
__device__ inline void lds_gravity_all(const HP &P, ClusterLds<NMAX> &C, int n, long long &pairs) {
    const JData J{C.pos, C.vel, C.mass, C.rinv, C.id};
    for (int i = (int)threadIdx.x; i < n; i += T) {
        double x[3], v[3], as[3], js[3], ad[3], jd[3];
        ld3(C.pos, i, x);
        ld3(C.vel, i, v);
        star_acc_jerk(P, x, v, as, js, nullptr);
        gravity_loop(P, J, n, C.id[i], x, v, C.rinv[i], ad, jd, nullptr);
        st3(C.acc_s, i, as);
        st3(C.jerk_s, i, js);
        st3(C.acc_d, i, ad);
        st3(C.jerk_d, i, jd);
        pairs += n - 1;
    }
}

// The unordered pairs {a, c} of the collision test (hermite.h:98-196): c = (a + d) mod n for
// d = 1 .. (n - 1) / 2 and every a, and for even n d = n / 2 with a < n / 2; thread t takes a
// = t mod n and every (T / n)-th distance.
template <int NMAX, class F>
__device__ inline void lds_pairs(int n, int a, int run, int runs, F pair) {
    if (run >= runs) return;
    const int h = (n - 1) >> 1;
    for (int d = 1 + run; d <= h; d += runs) pair(a + d < n ? a + d : a + d - n);
    if (!(n & 1) && run == runs - 1 && a < (n >> 1)) pair(a + (n >> 1));
}
// Whether one of this thread's pairs may have R < 1 (fr is NaN for the dead: false).  Every
// thread takes the same number of distances 1 .. n / 2 (the last again past the end, for even
// n the pairs at n / 2 twice), so that the loads of several are in flight together.
template <int NMAX>
__device__ inline bool lds_any_close(const ClusterLds<NMAX> &C, int n, int a, int run, int runs, int rounds) {
    const double fra = C.fr[a], xa = C.xp[3 * a], ya = C.xp[3 * a + 1], za = C.xp[3 * a + 2];
    bool close = false;
#pragma unroll 4
    for (int u = 0, d = 1 + run; u < rounds; u++, d += runs) {
        const int e = a + min(d, n >> 1), c = e < n ? e : e - n;
        const double dx = xa - C.xp[3 * c], dy = ya - C.xp[3 * c + 1], dz = za - C.xp[3 * c + 2];
        const double r2 = fra + C.fr[c];
        close |= dot3(dx, dy, dz, dx, dy, dz) < COL_FILTER * r2 * r2;
    }
    return close && n > 1;
}

// The collision of this block step, if any pair has R = |dx| / (f_i R_i + f_j R_j) < 1
// (hermite.h:98-196, 289-296): the pair with the smallest R (R is symmetric bit for bit, so
// the (R, lower, higher index) minimum is the first minimum of the reference's loops), the
// lighter body the impactor ic; every live member becomes a body, corrected to t_s.
template <int NMAX, int T>
__device__ bool lds_collide(ClusterLds<NMAX> &C, int n, double t_s, int a, int run, int runs, int &ic, int &jc) {
    const int t = (int)threadIdx.x, w = t >> 6;
    double rmin = 1.;
    int bi = 0x7fffffff, bj = 0x7fffffff;
    const double fra = C.fr[a], xa = C.xp[3 * a], ya = C.xp[3 * a + 1], za = C.xp[3 * a + 2];
    lds_pairs<NMAX>(n, a, run, runs, [&](int c) {
        const double dx = xa - C.xp[3 * c], dy = ya - C.xp[3 * c + 1], dz = za - C.xp[3 * c + 2];
        const double d2 = dot3(dx, dy, dz, dx, dy, dz);
        const double r2 = fra + C.fr[c];
        if (!(d2 < COL_FILTER * r2 * r2)) return;
        const double Rr = sqrt(d2) / r2;
        const int lo = min(a, c), hi = max(a, c);
        if (Rr < 1. && rlh_less(Rr, lo, hi, rmin, bi, bj)) { rmin = Rr; bi = lo; bj = hi; }
    });
    for (int d = 32; d > 0; d >>= 1) {
        const double ov = __shfl_xor(rmin, d);
        const int ol = __shfl_xor(bi, d), oh = __shfl_xor(bj, d);
        if (rlh_less(ov, ol, oh, rmin, bi, bj)) { rmin = ov; bi = ol; bj = oh; }
    }
    if ((t & 63) == 0) { C.red_r[w] = rmin; C.red_lo[w] = bi; C.red_hi[w] = bj; }
    __syncthreads();
    double rm = C.red_r[0];
    int gi = C.red_lo[0], gj = C.red_hi[0];
    for (int u = 1; u < T / 64; u++)
        if (rlh_less(C.red_r[u], C.red_lo[u], C.red_hi[u], rm, gi, gj)) {
            rm = C.red_r[u];
            gi = C.red_lo[u];
            gj = C.red_hi[u];
        }
    if (!(rm < 1.)) return false;
    if (C.mass[gi] < C.mass[gj]) { ic = gi; jc = gj; } else { ic = gj; jc = gi; }
    for (int i = t; i < n; i += T) C.dt[i] = t_s - C.time[i];
    __syncthreads();
    if (w == T / 64 - 1) lds_bodies(C, n, t_s, true);
    __syncthreads();
    return true;
}

// Perfect merging and its aftermath (hermite.h:449-458): everybody's force, the merged
// targets' acc/jerk, the initial block step of the live members, the twins' steps.  V: C's
// arrays for perfect_merge and merge_acc_jerk.
template <int NMAX, int T>
__device__ inline void lds_merge(const HP &P, ClusterLds<NMAX> &C, HardView &V, int n, int ic, int jc, double &ed,
                                 long long &pairs) {
    const int t = (int)threadIdx.x;
    if (t == 0) ed += perfect_merge(P, V, 0, n, ic, jc);
    __syncthreads();
    lds_gravity_all<NMAX, T>(P, C, n, pairs);
    __syncthreads();
    for (int i = t; i < n; i += T)
        if (C.flags[i] & GPLUM_FLAG_MERGED) merge_acc_jerk(V, 0, n, i);
    __syncthreads();
    for (int i = t; i < n; i += T)
        if (!(C.flags[i] & GPLUM_FLAG_DEAD)) {
            double ad[3], jd[3], as[3], js[3];
            ld3(C.acc_d, i, ad);
            ld3(C.jerk_d, i, jd);
            ld3(C.acc_s, i, as);
            ld3(C.jerk_s, i, js);
            C.dt[i] = dt_initial(P, C.time[i], C.dt[i], C.acc0[i], ad, jd, as, js);
        }
    lds_relations<NMAX, T>(C, n);
    __syncthreads();
    for (int i = t; i < n; i += T)
        if (C.twin_of[i] >= 0) C.dt[i] = C.dt[C.twin_of[i]];
    __syncthreads();
}

// mergeAccJerk (hermite.h:36-74) of component k: the mass-weighted mean of the hard force
// over target tt and its twins in ascending index, from the bodies' forces in C.fa
template <int NMAX>
__device__ inline void lds_family(const ClusterLds<NMAX> &C, int tt, int k, double &ad, double &jd) {
    double mass = C.mass[tt];
    int s = C.slot_of[tt];
    double sa = mass * C.fa[6 * s + k], sj = mass * C.fa[6 * s + 3 + k];
    for (int j = C.first[tt]; j >= 0; j = C.next[j]) {
        s = C.slot_of[j];
        sa += C.mass[j] * C.fa[6 * s + k];
        sj += C.mass[j] * C.fa[6 * s + 3 + k];
        mass += C.mass[j];
    }
    const double minv = 1. / mass;
    ad = sa * minv;
    jd = sj * minv;
}

// The pair terms of bodies c0 .. c0 + cb - 1 with every partner, one per thread (body c0 +
// my_r, partner my_j), into the three planes of s_term: (acc, jerk) by component, a row of
// np per body.  A partner with the body's own id (itself, a twin) gives +0, which leaves a
// sum begun at +0 unchanged.  Rows are padded with +0 to whole eights (lds_row), and their
// odd length and the planes' 4 mod 16 elements keep the quads' reads free of bank conflicts.
__host__ __device__ constexpr int lds_row(int n) { return ((n + 7) & ~7) + 1; }
constexpr int lds_plane(int slots) { return ((slots + 11) & ~15) + 4; }
// elements of a plane for clusters of nmin .. nmax members on T threads: a round holds T / n
// bodies, and there are n at most
constexpr int lds_terms(int T, int nmin, int nmax) {
    int m = 0;
    for (int n = nmin; n <= nmax; n++) {
        const int rows = T / n < n ? T / n : n;
        m = rows * lds_row(n) > m ? rows * lds_row(n) : m;
    }
    return lds_plane(m);
}
struct TermBody {          // what a thread holds of its body
    int slot, bd;
    double rinv;
    bool use, tv;
};
template <int NMAX>
__device__ inline TermBody lds_term_body(const ClusterLds<NMAX> &C, int c0, int nb, int cb, int my_r, int64_t idj) {
    TermBody B;
    const int s = c0 + my_r;
    B.tv = my_r < cb && s < nb;
    B.slot = B.tv ? s : 0;
    B.bd = C.body[B.slot];
    B.rinv = C.rinv[B.bd];
    B.use = C.id[B.bd] != idj;
    return B;
}
template <int NMAX, int T, int TP>
__device__ inline void lds_pair_terms(const HP &P, const ClusterLds<NMAX> &C, double2 *s_term, const TermBody &B,
                                      bool first, int row, const double xj[3], const double vj[3], double mj, double rj) {
    if (T > 64 && !__ballot(B.tv)) return;
    const double *px = first ? C.xp + 3 * B.bd : C.bx + 3 * B.slot;
    const double *pv = first ? C.vp + 3 * B.bd : C.bv + 3 * B.slot;
    const double xi[3] = {px[0], px[1], px[2]}, vi[3] = {pv[0], pv[1], pv[2]};
    double ta[3], tj[3];
    pair_term(P, xi, vi, B.rinv, xj[0], xj[1], xj[2], vj[0], vj[1], vj[2], mj, rj, ta, tj, nullptr,
              B.tv && B.use);
    if (B.tv)
        for (int d = 0; d < 3; d++) s_term[d * TP + row] = make_double2(B.use ? ta[d] : 0., B.use ? tj[d] : 0.);
}

// Predicts every member to t_s and lists the bodies of the block step.
template <int NMAX, int T>
__device__ inline void lds_predict(ClusterLds<NMAX> &C, int n, double t_s) {
    const int t = (int)threadIdx.x;
    for (int u = t; u < 3 * n; u += T)
        predict_one(t_s - C.time[u / 3], C.pos[u], C.vel[u], C.acc_s[u], C.jerk_s[u], C.acc_d[u], C.jerk_d[u], C.xp[u],
                    C.vp[u]);
    if (t >= T - 64) lds_bodies(C, n, t_s, false);
    if (t == 0) C.hit = 0;
    __syncthreads();
}

// A target's new time and step, and its twins'.
template <int NMAX>
__device__ inline void lds_advance(ClusterLds<NMAX> &C, int body, int fl, double t_c, double time, double dt,
                                   bool set_dt) {
    C.time[body] = time;
    if (set_dt) C.dt[body] = dt;
    if (fl & GPLUM_FLAG_MERGED)
        for (int j = C.first[body]; j >= 0; j = C.next[j]) {
            C.time[j] += t_c;
            if (set_dt) C.dt[j] = dt;
        }
}

// Block steps from (sys_time, loop) to the end of the soft step on the state in C, for
// clusters up to HARD_SEQ_MAX: the quads' state in registers, the hard force of a body
// summed sequentially in j.  Every thread of the workgroup calls it.
template <int NMAX, int T, int TP>
__device__ void integrate_seq(const HP &P, ClusterLds<NMAX> &C, HardView &V, double2 *s_term, int n, double &sys_time,
                              long long &loop, double &ed, int &n_col, long long &pairs) {
    constexpr int W = T / 64;
    static_assert(4 * NMAX <= T, "a quad per member");
    const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
    // quads from the last wave down, terms from the first wave up: with few bodies the two
    // run on different waves
    const int q = ((W - 1 - w) << 4) + (lane >> 2), k = lane & 3;
    const bool pad = k == 3;
    const int cb = T / n;                                   // bodies per round of terms
    const int my_r = t / n, my_j = t - my_r * n;            // this thread's body of a round, partner
    const int rounds = ((n >> 1) + cb - 1) / cb;            // distances per thread of the collision test
    const int np = lds_row(n);
    const double time_end = P.dt_tree;
    double t_s = lds_next_time(C, n);
    for (int u = t; u < 3 * TP; u += T) s_term[u] = make_double2(0., 0.);   // the rows' padding stays +0
    __syncthreads();
    int64_t idj = C.id[my_j];                               // changes with mergers only
    while (sys_time < time_end && loop < BLOCK_STEP_CAP) {
        lds_predict<NMAX, T>(C, n, t_s);
        double xj[3], vj[3];
        ld3(C.xp, my_j, xj);
        ld3(C.vp, my_j, vj);
        const double mj = C.mass[my_j], rj = C.rinv[my_j];
        int flag_col = 0, ic = -1, jc = -1, nb = 0, anym = 0, body = 0, tt = 0, fl = 0;
        double time_b = 0., dt_b = 0., acc0_b = 0.;
        TermBody B;
        bool on = false;                                    // this quad holds a body
        double xp = 0., vp = 0., a0s = 0., j0s = 0., a0d = 0., j0d = 0., t_c = 0.;
        double x = 0., v = 0., as = 0., js = 0., ad = 0., jd = 0., a2s = 0., a3s = 0., a2d = 0., a3d = 0.;

        // acc/jerk (Sun: as, js; hard: ad, jd) of the bodies at the predicted (first) or
        // corrected state, in their quads' lanes
        auto evaluate = [&](bool first) {
            if (W == 1 || ((W - 1 - w) << 4) < nb) star_quad(P, x, v, pad, as, js);
            if (first && !flag_col && P.collision) {
                if (lds_any_close(C, n, my_j, my_r, cb, rounds)) C.hit = 1;
            }
            if (nb == 0) __syncthreads();     // no step left to take (steps that are not numbers)
            for (int c0 = 0; c0 < nb; c0 += cb) {
                if (c0) {
                    const TermBody D = lds_term_body(C, c0, nb, cb, my_r, idj);
                    lds_pair_terms<NMAX, T, TP>(P, C, s_term, D, first, my_r * np + my_j, xj, vj, mj, rj);
                } else {
                    lds_pair_terms<NMAX, T, TP>(P, C, s_term, B, first, my_r * np + my_j, xj, vj, mj, rj);
                }
                __syncthreads();
                if (q >= c0 && q < min(nb, c0 + cb) && !pad) {
                    const double2 *p = s_term + k * TP + (q - c0) * np;
                    ad = 0.;
                    jd = 0.;
                    // eight in flight while the last eight are added
                    double2 u[8], z[8];
                    auto load = [&](double2 (&e)[8], int j) __attribute__((always_inline)) {
#pragma unroll
                        for (int m = 0; m < 8; m++) e[m] = p[j + m];
                    };
                    auto add = [&](const double2 (&e)[8]) __attribute__((always_inline)) {
#pragma unroll
                        for (int m = 0; m < 8; m++) {
                            ad += e[m].x;
                            jd += e[m].y;
                        }
                    };
                    load(u, 0);
                    for (int j = 8;; j += 16) {
                        if (j >= n) { add(u); break; }
                        load(z, j);
                        add(u);
                        if (j + 8 >= n) { add(z); break; }
                        load(u, j + 8);
                        add(z);
                    }
                }
                if (c0 + cb < nb) __syncthreads();
            }
            if (anym) {
                if (on && !pad) {
                    C.fa[6 * q + k] = ad;
                    C.fa[6 * q + 3 + k] = jd;
                }
                __syncthreads();
                if (on && !pad && (fl & GPLUM_FLAG_MERGED)) lds_family(C, tt, k, ad, jd);
            }
        };

        for (;;) {
            nb = C.nb;
            anym = C.anym;
            on = q < nb;
            body = on ? C.body[q] : 0;
            tt = C.twin_of[body] >= 0 ? C.twin_of[body] : body;
            const int u = 3 * body + (pad ? 0 : k);
            xp = pad ? 0. : C.xp[u];
            vp = pad ? 0. : C.vp[u];
            a0s = pad ? 0. : C.acc_s[u];
            j0s = pad ? 0. : C.jerk_s[u];
            a0d = pad ? 0. : C.acc_d[u];
            j0d = pad ? 0. : C.jerk_d[u];
            time_b = C.time[tt];
            dt_b = C.dt[body];
            acc0_b = C.acc0[body];
            fl = C.flags[tt];
            B = lds_term_body(C, 0, nb, cb, my_r, idj);
            t_c = t_s - time_b;
            x = xp;
            v = vp;
            evaluate(true);
            if (flag_col || !P.collision || !C.hit || !lds_collide<NMAX, T>(C, n, t_s, my_j, my_r, cb, ic, jc)) break;
            flag_col = 1;
        }
        // two corrections (hermite.h:300-375)
        const double Dt2 = t_c * t_c;
        const double Dt_inv = recip_step(t_c);
        const double Dt_inv2 = Dt_inv * Dt_inv;
        const double Dt_inv3 = Dt_inv2 * Dt_inv;
        for (int ite = 0; ite < 2; ite++) {
            if (on) {
                correct_one(t_c, Dt2, Dt_inv2, Dt_inv3, xp, vp, as, a0s, j0s, js, ad, a0d, j0d, jd, x, v, a2s, a3s, a2d,
                            a3d);
                if (!pad) {
                    C.bx[3 * q + k] = x;
                    C.bv[3 * q + k] = v;
                }
            }
            __syncthreads();
            evaluate(false);
        }
        if (on) {
            const bool target = tt == body;
            const double time = time_b + t_c;
            double dt = dt_b;
            if (!flag_col && target) dt = dt_block_quad(P, time, dt, acc0_b, ad, jd, a2d, a3d, as, js, a2s, a3s);
            if (!pad) {
                const int u = 3 * body + k;
                C.pos[u] = x;
                C.vel[u] = v;
                C.acc_s[u] = as;
                C.jerk_s[u] = js;
                C.acc_d[u] = ad;
                C.jerk_d[u] = jd;
            }
            if (k == 0) {
                pairs += 3 * (long long)(n - 1);
                if (target) lds_advance(C, body, fl, t_c, time, dt, !flag_col);
            }
        }
        __syncthreads();
        if (flag_col) {
            lds_merge<NMAX, T>(P, C, V, n, ic, jc, ed, pairs);
            idj = C.id[my_j];
            n_col++;
        }
        t_s = lds_next_time(C, n);
        sys_time = lds_system_time(C, n, t_s, time_end, sys_time);
        loop++;
    }
}

// The same for the clusters above HARD_SEQ_MAX, whose hard forces are summed as 64
// lane-strided partials and a butterfly (coop_pair_sum): a wave per body, so that the partials
// need no LDS.  More members than quads: a quad takes the bodies q, q + T / 4, ..., whose
// state stays in LDS between the phases.

// The butterfly of coop_pair_sum over six values at once: the additions are the same pairs,
// but the rows of 16 lanes (the halves, at distance 32) each keep some of the components,
// exchanged by lane swaps: 9 + 8 + 28 instructions for the levels 32, 16 and 8 to 1 where six
// separate butterflies take about 130.  Lane 0 of row r ends with component {0, 1, 3, 4}[r] in
// A; rows 0 and 2 with components 2 and 5 in B.
__device__ inline double swap_add32(double x, double y) {     // x + x(lane ^ 32) below lane 32, y's above
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return dbl_of(lo[0], hi[0]) + dbl_of(lo[1], hi[1]);
}
__device__ inline double swap_add16(double x, double y) {     // x + x(lane ^ 16) in even rows, y's in odd ones
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return dbl_of(lo[0], hi[0]) + dbl_of(lo[1], hi[1]);
}
__device__ inline void butterfly6(const double a[3], const double j[3], double &A, double &B) {
    const double v0 = swap_add32(a[0], j[0]), v1 = swap_add32(a[1], j[1]), v2 = swap_add32(a[2], j[2]);
    A = swap_add16(v0, v1);
    B = swap_add16(v2, v2);
    A += dpp_f64<DPP_ROW_ROR8>(A);
    B += dpp_f64<DPP_ROW_ROR8>(B);
    A += dpp_f64<DPP_QUAD_3210>(dpp_f64<DPP_ROW_HALF_MIRROR>(A));
    B += dpp_f64<DPP_QUAD_3210>(dpp_f64<DPP_ROW_HALF_MIRROR>(B));
    A += dpp_f64<DPP_QUAD_2301>(A);
    B += dpp_f64<DPP_QUAD_2301>(B);
    A += dpp_f64<DPP_QUAD_1032>(A);
    B += dpp_f64<DPP_QUAD_1032>(B);
}

template <int NMAX>
struct TreeLds {
    double sa[6 * NMAX];               // the Sun's acc/jerk of the bodies (by slot)
    double a23[12 * NMAX];             // a2_s, a3_s, a2_d, a3_d of the last correction (by slot)
};

template <int NMAX, int T>
__device__ void integrate_tree(const HP &P, ClusterLds<NMAX> &C, TreeLds<NMAX> &E, HardView &V, int n, double &sys_time,
                               long long &loop, double &ed, int &n_col, long long &pairs) {
    constexpr int W = T / 64, NQ = T / 4;
    const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
    const int q = ((W - 1 - w) << 4) + (lane >> 2), k = lane & 3;
    const bool pad = k == 3;
    const int cb = T / n;
    const int my_r = t / n, my_j = t - my_r * n;
    const int rounds = ((n >> 1) + cb - 1) / cb;
    const double time_end = P.dt_tree;
    double t_s = lds_next_time(C, n);
    while (sys_time < time_end && loop < BLOCK_STEP_CAP) {
        lds_predict<NMAX, T>(C, n, t_s);
        int flag_col = 0, ic = -1, jc = -1, nb = 0;

        auto evaluate = [&](bool first) {
            for (int s = q; s < nb; s += NQ) {
                const int u = first ? 3 * C.body[s] : 3 * s;
                const double x = pad ? 0. : (first ? C.xp : C.bx)[u + k], v = pad ? 0. : (first ? C.vp : C.bv)[u + k];
                double as, js;
                star_quad(P, x, v, pad, as, js);
                if (!pad) {
                    E.sa[6 * s + k] = as;
                    E.sa[6 * s + 3 + k] = js;
                }
            }
            if (first && !flag_col && P.collision) {
                if (lds_any_close(C, n, my_j, my_r, cb, rounds)) C.hit = 1;
            }
            const JData J{C.xp, C.vp, C.mass, C.rinv, C.id};
            for (int s = w; s < nb; s += W) {
                const int bd = C.body[s];
                const double *px = first ? C.xp + 3 * bd : C.bx + 3 * s;
                const double *pv = first ? C.vp + 3 * bd : C.bv + 3 * s;
                const double xi[3] = {px[0], px[1], px[2]}, vi[3] = {pv[0], pv[1], pv[2]};
                double a[3] = {0., 0., 0.}, jk[3] = {0., 0., 0.}, A, B;
                const int64_t id = C.id[bd];
                const double rinv = C.rinv[bd];
                // the lane's partial: j = lane, lane + 64, ..., two at a time (past the end the
                // last member again, not added)
                for (int j0 = 0; j0 < n; j0 += 128) {
                    double ta[2][3], tj[2][3];
                    bool use[2];
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const int j = min(j0 + 64 * u + lane, n - 1);
                        use[u] = j0 + 64 * u + lane < n && C.id[j] != id;
                        pair_term_j(P, J, j, xi, vi, rinv, ta[u], tj[u], nullptr, use[u]);
                    }
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        for (int d = 0; d < 3; d++) {
                            a[d] = use[u] ? a[d] + ta[u][d] : a[d];
                            jk[d] = use[u] ? jk[d] + tj[u][d] : jk[d];
                        }
                }
                butterfly6(a, jk, A, B);
                if ((lane & 15) == 0) {
                    const int r = lane >> 4;
                    C.fa[6 * s + (r < 2 ? r : r + 1)] = A;
                    if (!(r & 1)) C.fa[6 * s + 2 + 3 * (r >> 1)] = B;
                }
            }
            __syncthreads();
        };
        // the hard force of slot s, component k (after mergeAccJerk)
        auto hard_force = [&](int s, int tt, double &ad, double &jd) {
            ad = C.fa[6 * s + k];
            jd = C.fa[6 * s + 3 + k];
            if (C.flags[tt] & GPLUM_FLAG_MERGED) lds_family(C, tt, k, ad, jd);
        };

        for (;;) {
            nb = C.nb;
            evaluate(true);
            if (flag_col || !P.collision || !C.hit || !lds_collide<NMAX, T>(C, n, t_s, my_j, my_r, cb, ic, jc)) break;
            flag_col = 1;
        }
        for (int ite = 0; ite < 2; ite++) {
            for (int s = q; s < nb; s += NQ) {
                const int body = C.body[s], tt = C.twin_of[body] >= 0 ? C.twin_of[body] : body;
                const int u = 3 * body + k;
                if (pad) continue;
                double ad, jd, x, v, a2s, a3s, a2d, a3d;
                hard_force(s, tt, ad, jd);
                const double t_c = t_s - C.time[tt];
                const double Dt_inv = recip_step(t_c);
                const double Dt_inv2 = Dt_inv * Dt_inv;
                correct_one(t_c, t_c * t_c, Dt_inv2, Dt_inv2 * Dt_inv, C.xp[u], C.vp[u], E.sa[6 * s + k], C.acc_s[u],
                            C.jerk_s[u], E.sa[6 * s + 3 + k], ad, C.acc_d[u], C.jerk_d[u], jd, x, v, a2s, a3s, a2d, a3d);
                C.bx[3 * s + k] = x;
                C.bv[3 * s + k] = v;
                if (ite == 1) {
                    double *z = E.a23 + 12 * s + k;
                    z[0] = a2s;
                    z[3] = a3s;
                    z[6] = a2d;
                    z[9] = a3d;
                }
            }
            __syncthreads();
            evaluate(false);
        }
        for (int s = q; s < nb; s += NQ) {
            const int body = C.body[s], tt = C.twin_of[body] >= 0 ? C.twin_of[body] : body;
            const bool target = tt == body;
            double ad = 0., jd = 0., as = 0., js = 0., a2s = 0., a3s = 0., a2d = 0., a3d = 0.;
            if (!pad) {
                hard_force(s, tt, ad, jd);
                as = E.sa[6 * s + k];
                js = E.sa[6 * s + 3 + k];
                const double *z = E.a23 + 12 * s + k;
                a2s = z[0];
                a3s = z[3];
                a2d = z[6];
                a3d = z[9];
                const int u = 3 * body + k;
                C.pos[u] = C.bx[3 * s + k];
                C.vel[u] = C.bv[3 * s + k];
                C.acc_s[u] = as;
                C.jerk_s[u] = js;
                C.acc_d[u] = ad;
                C.jerk_d[u] = jd;
            }
            if (k == 0) pairs += 3 * (long long)(n - 1);
            if (!target) continue;            // a twin takes its target's time and step
            const double t_c = t_s - C.time[body], time = C.time[body] + t_c;
            double dt = C.dt[body];
            if (!flag_col) dt = dt_block_quad(P, time, dt, C.acc0[body], ad, jd, a2d, a3d, as, js, a2s, a3s);
            if (k == 0) lds_advance(C, body, C.flags[body], t_c, time, dt, !flag_col);
        }
        __syncthreads();
        if (flag_col) {
            lds_merge<NMAX, T>(P, C, V, n, ic, jc, ed, pairs);
            n_col++;
        }
        t_s = lds_next_time(C, n);
        sys_time = lds_system_time(C, n, t_s, time_end, sys_time);
        loop++;
    }
}

// One cluster [b, b + n) of H: loaded into C, integrated, the final calcGravity with
// potentials (hermite.h:466-470), written back.  fresh: from the start of the soft step,
// with the initial calcGravity (hermite.h:259-270); else from the block step a faster path
// stopped at, whose state is in H.
// integrate: the block steps (integrate_seq or integrate_tree).
template <int NMAX, int T, class F>
__device__ __forceinline__ void run_cluster_lds(const HP &P, HardView &H, ClusterLds<NMAX> &C, int b, int n, bool fresh,
                                                int &n_col, long long &pairs, F integrate) {
    const int t = (int)threadIdx.x;
    for (int u = t; u < 3 * n; u += T) {
        C.pos[u] = H.pos[3 * b + u];
        C.vel[u] = H.vel[3 * b + u];
        C.acc_s[u] = H.acc_s[3 * b + u];
        C.jerk_s[u] = H.jerk_s[3 * b + u];
        C.acc_d[u] = H.acc_d[3 * b + u];
        C.jerk_d[u] = H.jerk_d[3 * b + u];
    }
    for (int i = t; i < n; i += T) {
        C.mass[i] = H.mass[b + i];
        C.rinv[i] = H.rinv[b + i];
        C.time[i] = H.time[b + i];
        C.dt[i] = H.dt[b + i];
        C.acc0[i] = H.acc0[b + i];
        C.r_planet[i] = H.r_planet[b + i];
        C.f[i] = H.f[b + i];
        C.id[i] = H.id[b + i];
        C.flags[i] = H.flags[b + i] & ~(GPLUM_FLAG_DEAD | GPLUM_FLAG_MERGED);
        C.twin_of[i] = -1;
    }
    __syncthreads();
    lds_relations<NMAX, T>(C, n);
    if (fresh) {
        long long none = 0;                 // the caller counts the initial evaluation
        lds_gravity_all<NMAX, T>(P, C, n, none);
    }
    __syncthreads();
    HardView V = H;
    V.pos = C.pos; V.vel = C.vel; V.acc_s = C.acc_s; V.jerk_s = C.jerk_s; V.acc_d = C.acc_d; V.jerk_d = C.jerk_d;
    V.mass = C.mass; V.rinv = C.rinv; V.time = C.time; V.dt = C.dt; V.acc0 = C.acc0; V.r_planet = C.r_planet;
    V.f = C.f; V.id = C.id; V.flags = C.flags; V.twin_of = C.twin_of;
    V.base = b;
    integrate(V);
    const JData J{C.pos, C.vel, C.mass, C.rinv, C.id};
    for (int i = t; i < n; i += T) {
        double x[3], v[3], as[3], js[3], ad[3], jd[3], phs = 0., phd = 0.;
        ld3(C.pos, i, x);
        ld3(C.vel, i, v);
        star_acc_jerk(P, x, v, as, js, &phs);
        gravity_loop(P, J, n, C.id[i], x, v, C.rinv[i], ad, jd, &phd);
        pairs += n - 1;
        H.phi_s[b + i] = phs;
        H.phi_d[b + i] = phd;
        st3(C.acc_s, i, as);
        st3(C.jerk_s, i, js);
        st3(C.acc_d, i, ad);
        st3(C.jerk_d, i, jd);
    }
    __syncthreads();
    if (n_col > 0) {
        for (int i = t; i < n; i += T)
            if (C.flags[i] & GPLUM_FLAG_MERGED) merge_acc_jerk(V, 0, n, i);
        __syncthreads();
    }
    for (int u = t; u < 3 * n; u += T) {
        H.pos[3 * b + u] = C.pos[u];
        H.vel[3 * b + u] = C.vel[u];
        H.acc_s[3 * b + u] = C.acc_s[u];
        H.jerk_s[3 * b + u] = C.jerk_s[u];
        H.acc_d[3 * b + u] = C.acc_d[u];
        H.jerk_d[3 * b + u] = C.jerk_d[u];
    }
    for (int i = t; i < n; i += T) {
        H.time[b + i] = C.time[i];
        H.dt[b + i] = C.dt[i];
        H.r_planet[b + i] = C.r_planet[i];
        H.id[b + i] = C.id[i];
        H.flags[b + i] = C.flags[i];
        H.twin_of[b + i] = C.twin_of[i];
    }
    __syncthreads();
}

}  // namespace gplum
