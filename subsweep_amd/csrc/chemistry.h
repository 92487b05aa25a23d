// FP64 hydrogen-only chemistry for one cell (device and host), after
// HydrogenOnly / Solver in src/chemistry/hydrogen_only/mod.rs:68-461.
//
// Rates are the Rosdahl et al. (2015) fits the reference uses; operation order
// follows the reference expression by expression (no FMA contraction: the
// library is compiled with -ffp-contract=off). The recursive sub-stepping of
// perform_timestep_internal (:394-424) is run as an explicit depth-first walk:
// a rejected step of depth k is replaced by two steps of depth k+1; the second
// one is remembered as a bit in `pending` (at most one per depth can be
// outstanding), and the walk always resumes at the deepest pending step. The
// returned timescale is the one of the last accepted step, as in the reference.
#pragma once

#include <cfloat>
#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#define SSW_HD __host__ __device__ inline
#else
#define SSW_HD inline
#endif

namespace ssw {

// Unit factors and constants, src/units/mod.rs:19-108 (products as diman forms them).
constexpr double kCm = 0.01;
constexpr double kCm2 = kCm * kCm;
constexpr double kCm3 = 1e-6;
constexpr double kCm3PerS = kCm3 / 1.0;
constexpr double kErg = 1e-7 * 1.0;
constexpr double kErgCm3PerS = kErg * kCm3PerS;
constexpr double kErgPerS = kErg / 1.0;
constexpr double kEv = 1.602176634e-19 * 1.0;
constexpr double kBoltzmann = 1.380649e-23 * 1.0 / 1.0;
constexpr double kProtonMass = 1.67262192369e-27;
constexpr double kGamma = 5.0 / 3.0;
constexpr double kSigma = 2.9580524545305314e-18 * kCm2;  // NUMBER_WEIGHTED_AVERAGE_CROSS_SECTION
constexpr double kPhotonEnergy = 18.028356312818811 * kEv;
constexpr double kRydberg = 13.65693 * kEv;
constexpr double kXEps = 1e-10;             // IONIZED_HYDROGEN_FRACTION_EPSILON
constexpr double kInvEps = 1.0 / DBL_EPSILON;  // 1.0 / f64::EPSILON
constexpr int kMaxDepth = 100;

enum { kProcTemperature = 0, kProcIonization = 1, kProcPhotonRate = 2 };

// f64::powi lowered by LLVM to binary exponentiation.
SSW_HD double powi(double a, int b) {
    bool recip = b < 0;
    double r = 1.0;
    for (;;) {
        if (b & 1) r *= a;
        b /= 2;
        if (b == 0) break;
        a *= a;
    }
    return recip ? 1.0 / r : r;
}

// Attenuation of one cell: exp(-(rho/m_p (1-x)) sigma L), the non-absorbed
// fraction of HydrogenOnly::get_outgoing_rate (hydrogen_only/mod.rs:78-86).
SSW_HD double non_absorbed_fraction(double density, double xhii, double size) {
    double n = density / kProtonMass * (1.0 - xhii);
    return exp(-n * kSigma * size);
}

struct Cell {
    double x, T;              // ionised fraction, temperature
    double rho, vol, len, rate, a;
};

// --- rate fits (hydrogen_only/mod.rs:161-302) ---------------------------------
// The fits take the exponentials and powers they contain as arguments, so that
// a solver step gathers them and evaluates them together (transcendentals
// below): they are nearly all of its time, and on the device the lanes of a
// quad share them.
SSW_HD double fit_collision(double t, double e) {  // e = exp(-157809.1 / t)
    return sqrt(t) / (1.0 + sqrt(t / 1e5)) * e;
}
SSW_HD double fit_collision_dt(double t, double e) {
    const double k1 = 1.0 / 1e5, k2 = 157809.1;
    double s = sqrt(k1 * t);
    return (e * (k1 * k2 * t + 0.5 * s * (2.0 * k2 + t))) /
           (sqrt(powi(t, 3)) * s * powi(s + 1.0, 2));
}
// alpha_B: l15 = l^1.5, w = (1 + (l / 2.74)^0.407)^2.242 with l = 315614 / T
SSW_HD double alpha_b(double l15, double w) { return (2.753e-14 * l15 / w) * kCm3PerS; }
// p = (k1 l)^0.407, w = (p + 1)^(-3.242)
SSW_HD double alpha_b_dt(double T, double p, double w) {
    double l = 315614.0 / T;
    double dl = -315614.0 / (T * T);
    const double k2 = 0.407, k3 = 2.242;
    double d = -sqrt(l) * w * (k2 * k3 * p - 1.5 * p - 1.5);
    return ((2.753e-14 * d) * kCm3PerS) * dl;
}
// l197 = l^1.97, w = (1 + (l / 2.25)^0.376)^3.72
SSW_HD double recomb_cooling(double T, double l197, double w) {
    return (3.435e-30 * T * l197 / w) * kErgCm3PerS;
}
// q = (k1 / (k5 T))^0.376, w = (1 + q)^(-4.72)
SSW_HD double recomb_cooling_dt(double l197, double q, double w) {
    const double k2 = 1.97, k3 = 0.376, k4 = 3.72;
    double v = w * (1.0 - 1.0 * k2 + (1.0 - 1.0 * k2 + k3 * k4) * q) * l197;
    return ((3.435e-30 * v) * kErgCm3PerS) / 1.0;
}
SSW_HD double beta_ci(double T, double e) { return (5.85e-11 * fit_collision(T, e)) * kCm3PerS; }
SSW_HD double beta_ci_dt(double T, double e) { return ((5.85e-11 * fit_collision_dt(T, e)) * kCm3PerS) / 1.0; }
SSW_HD double ci_cooling(double T, double e) { return (1.27e-21 * fit_collision(T, e)) * kErgCm3PerS; }
SSW_HD double ci_cooling_dt(double T, double e) { return ((1.27e-21 * fit_collision_dt(T, e)) * kErgCm3PerS) / 1.0; }
SSW_HD double ce_cooling(double T, double e) {  // e = exp(-118348 / T)
    return (7.5e-19 / (1.0 + sqrt(T / 1e5)) * e) * kErgCm3PerS;
}
SSW_HD double ce_cooling_dt(double T, double e) {
    const double k1 = 7.5e-19, k2 = 118348.0, k3 = 1.0 / 1e5;
    double s = sqrt(k3 * T);
    double v = (k1 * e * (k2 * k3 * T - 0.5 * k3 * powi(T, 2) + k2 * s)) /
               (powi(T, 2) * s * powi(1.0 + s, 2));
    return (v * kErgCm3PerS) / 1.0;
}
SSW_HD double brems_cooling(double T) { return (1.42e-27 * sqrt(T)) * kErgCm3PerS; }
SSW_HD double brems_cooling_dt(double T) { return ((1.42e-27 / (2.0 * sqrt(T))) * kErgCm3PerS) / 1.0; }
SSW_HD double compton_cooling(double T, double a) {
    double x = 2.727 / a;
    return (1.017e-37 * powi(x, 4) * (T - x)) * kErgPerS;
}
SSW_HD double compton_cooling_dt(double a) {
    double x = 2.727 / a;
    return ((1.017e-37 * powi(x, 4)) * kErgPerS) / 1.0;
}

// --- derived quantities -----------------------------------------------------------
SSW_HD double n_h(const Cell& c) { return c.rho / kProtonMass; }
SSW_HD double n_hii(const Cell& c) { return n_h(c) * c.x; }
SSW_HD double n_hi(const Cell& c) { return n_h(c) * (1.0 - c.x); }
SSW_HD double mu(const Cell& c) { return 1.0 / (c.x + 1.0); }

// Powers and exponentials of up to four argument pairs at once: one after the
// other, or (Quad) one per lane of a quad.
struct Serial {
    template <int kN>
    SSW_HD void powers(const double (&b)[kN], const double (&e)[kN], double (&out)[kN]) const {
#pragma unroll
        for (int i = 0; i < kN; i++) out[i] = pow(b[i], e[i]);
    }
    template <int kN>
    SSW_HD void exps(const double (&a)[kN], double (&out)[kN]) const {
#pragma unroll
        for (int i = 0; i < kN; i++) out[i] = exp(a[i]);
    }
};

#if defined(__HIPCC__)
// The four lanes of a quad hold the same cell: each evaluates one of the
// arguments and all get the results (the same calls, so the same bits).
struct Quad {
    template <int kI>
    static __device__ __forceinline__ double from(double v) {  // lane kI's value, on every lane of the quad
        const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), kI * 0x55, 0xF, 0xF, true);
        const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), kI * 0x55, 0xF, 0xF, true);
        return __hiloint2double(hi, lo);
    }
    template <int kN>
    static __device__ __forceinline__ double mine(const double (&a)[kN]) {
        const unsigned r = threadIdx.x & 3u;
        double v = a[0];
#pragma unroll
        for (int i = 1; i < kN; i++) v = r == (unsigned)i ? a[i] : v;
        return v;
    }
    template <int kN>
    static __device__ __forceinline__ void share(double v, double (&out)[kN]) {
        static_assert(kN <= 4, "one argument per lane of a quad");
        out[0] = from<0>(v);
        if constexpr (kN > 1) out[1] = from<1>(v);
        if constexpr (kN > 2) out[2] = from<2>(v);
        if constexpr (kN > 3) out[3] = from<3>(v);
    }
    template <int kN>
    __device__ __forceinline__ void powers(const double (&b)[kN], const double (&e)[kN], double (&out)[kN]) const {
        share(pow(mine(b), mine(e)), out);
    }
    template <int kN>
    __device__ __forceinline__ void exps(const double (&a)[kN], double (&out)[kN]) const {
        share(exp(mine(a)), out);
    }
};
#endif

// What the temperature's step takes: cooling and its derivative at T, and the
// transmitted fraction of the cell (the ionised fraction's step has it too).
struct HeatRates {
    double ce, ci, pass;    // exp(-118348 / T), exp(-157809.1 / T), exp(-n_HI sigma L)
    double l197, w, q, wd;  // recomb_cooling's and recomb_cooling_dt's powers
};
struct IonRates {
    double ci;              // exp(-157809.1 / T)
    double l15, w, p, wd;   // alpha_b's and alpha_b_dt's powers
};

template <typename Ev>
SSW_HD HeatRates heat_rates(const Cell& c, const Ev& ev) {
    const double l = 315614.0 / c.T;
    const double k1 = 315614.0, k4 = 3.72, k5 = 2.25;
    double p[3], w[2], e[3];
    ev.template powers<3>({l, l / 2.25, k1 / (k5 * c.T)}, {1.97, 0.376, 0.376}, p);
    ev.template powers<2>({1.0 + p[1], 1.0 + p[2]}, {3.72, -1.0 - k4}, w);
    ev.template exps<3>({-118348.0 / c.T, -157809.1 / c.T, -n_hi(c) * kSigma * c.len}, e);
    return {e[0], e[1], e[2], p[0], w[0], p[2], w[1]};
}
template <typename Ev>
SSW_HD IonRates ion_rates(const Cell& c, const Ev& ev) {
    const double l = 315614.0 / c.T;
    const double k1 = 1.0 / 2.74, k3 = 2.242;
    double p[3], w[2], e[1];
    ev.template powers<3>({l, l / 2.74, k1 * l}, {1.5, 0.407, 0.407}, p);
    ev.template powers<2>({1.0 + p[1], p[2] + 1.0}, {2.242, -k3 - 1.0}, w);
    ev.template exps<1>({-157809.1 / c.T}, e);
    return {e[0], p[0], w[0], p[2], w[1]};
}

SSW_HD double cooling(const Cell& c, const HeatRates& r) {
    double ne = n_hii(c), n0 = n_hi(c), n1 = n_hii(c);
    double coll = (ce_cooling(c.T, r.ce) + ci_cooling(c.T, r.ci)) * ne * n0;
    double rec = recomb_cooling(c.T, r.l197, r.w) * ne * n1;
    double br = brems_cooling(c.T) * ne * n1;
    double co = compton_cooling(c.T, c.a) * ne;
    return coll + rec + br + co;
}
SSW_HD double cooling_dt(const Cell& c, const HeatRates& r) {
    double ne = n_hii(c), n0 = n_hi(c), n1 = n_hii(c);
    double coll = (ce_cooling_dt(c.T, r.ce) + ci_cooling_dt(c.T, r.ci)) * ne * n0;
    double rec = recomb_cooling_dt(r.l197, r.q, r.wd) * ne * n1;
    double br = brems_cooling_dt(c.T) * ne * n1;
    double co = compton_cooling_dt(c.a) * ne;
    return coll + rec + br + co;
}
SSW_HD double newly_ionized(const Cell& c, double dt, double pass) {  // :312-319
    double absorbed = 1.0 - pass;
    double photons = dt * c.rate;
    return photons * absorbed;
}
SSW_HD double delta_temperature(const Cell& c, double dt, const HeatRates& r) {  // :304-310
    double k = (kGamma - 1.0) * kProtonMass / (c.rho * kBoltzmann);
    double heat = newly_ionized(c, dt, r.pass) / c.vol * (kPhotonEnergy - kRydberg) / dt;  // photoheating_rate
    double lam = heat - cooling(c, r);
    double dlam = -cooling_dt(c, r);
    double m = mu(c);
    return k * m * lam * dt / (1.0 - k * m * dlam * dt);
}
SSW_HD double delta_ionized(const Cell& c, double dt, const IonRates& r, double pass) {  // :334-354 (Rosdahl+15 A23)
    double nh = n_h(c);
    double ne = n_hii(c);
    double al = alpha_b(r.l15, r.w), dal = alpha_b_dt(c.T, r.p, r.wd);
    double be = beta_ci(c.T, r.ci), dbe = beta_ci_dt(c.T, r.ci);
    double gam = newly_ionized(c, dt, pass) / (n_hi(c) * c.vol) / dt;  // photoionization_rate
    double cc = be * ne + gam;
    double m = mu(c);
    double dd = al * ne;
    double x = c.x;
    double rc = ne * c.T * m * 1.0 * dbe;
    double dcdx = nh * be - rc;
    double rd = ne * c.T * m * 1.0 * dal;
    double dddx = nh * al - rd;
    double j = dcdx - (cc + dd) - x * (dcdx + dddx);
    return dt * (cc - x * (cc + dd)) / (1.0 - j * dt);
}

// --- optional outputs of the solver (src/sweep/chemistry_output.rs:25-56) -------
// evaluated with the fixed timestep of :15-19 (1 yr = 3.15576e7 s,
// src/units/mod.rs:48) on the state after the step, without a floor
constexpr double kYear = 3.15576e7;
SSW_HD double photoionization_rate(const Cell& c, double dt, double pass) {  // hydrogen_only/mod.rs:327-332
    return newly_ionized(c, dt, pass) / (n_hi(c) * c.vol) / dt;
}
SSW_HD double photoheating_rate(const Cell& c, double dt, double pass) {  // :321-325
    return newly_ionized(c, dt, pass) / c.vol * (kPhotonEnergy - kRydberg) / dt;
}
// PhotoionizationRate, HeatingRate (photoheating - cooling), RecombinationRate
// (alpha_B n_e x), CollisionalIonizationRate (beta n_e (1 - x))
SSW_HD void chemistry_outputs(const Cell& c, double (&out)[4]) {
    const HeatRates h = heat_rates(c, Serial());
    const IonRates i = ion_rates(c, Serial());
    out[0] = photoionization_rate(c, kYear, h.pass);
    out[1] = photoheating_rate(c, kYear, h.pass) - cooling(c, h);
    out[2] = alpha_b(i.l15, i.w) * n_hii(c) * c.x;
    out[3] = beta_ci(c.T, i.ci) * n_hii(c) * (1.0 - c.x);
}

struct Floor {
    bool on;
    double T, x;
};

SSW_HD void clamp_state(Cell& c, const Floor& f) {  // :356-369
    double lo = f.on ? f.x : kXEps;
    double hi = 1.0 - kXEps;
    double v = c.x;
    if (v < lo) v = lo;
    if (v > hi) v = hi;
    c.x = v;
    if (f.on && c.T < f.T) c.T = f.T;
}

// update() of :444-461; false = TimestepCriterionViolated.
SSW_HD bool accept(double& value, double change, double safety, double dt, double& rec) {
    double rel = fmin(fabs(change / value), kInvEps);
    if (rel > safety) return false;
    value += change;
    rec = dt * (safety / rel);
    return true;
}

// try_timestep_update (:371-392) with the rates h at c
template <typename Ev>
SSW_HD bool try_step(Cell& c, const Floor& f, double dt, double safety, double& ts, int& proc, const HeatRates& h,
                     const Ev& ev) {
    double dT = delta_temperature(c, dt, h);
    double tsT;
    if (!accept(c.T, dT, safety, dt, tsT)) return false;
    double dx = delta_ionized(c, dt, ion_rates(c, ev), h.pass);
    double tsx;
    if (!accept(c.x, dx, safety, dt, tsx)) return false;
    clamp_state(c, f);
    if (tsT < tsx) {
        ts = tsT;
        proc = kProcTemperature;
    } else {
        ts = tsx;
        proc = kProcIonization;
    }
    return true;
}

// A cell's walk through its sub-steps: the pending second halves (bit =
// depth), the current depth and step, and the timescale and process of the
// last accepted step.
struct Walk {
    uint64_t lo = 0, hi = 0;
    int depth = 0;
    double dt = 0.0, ts = 0.0;
    int proc = kProcTemperature;
    bool failed = false;

    SSW_HD void overflow(double dt0) {
        failed = true;
        proc = kProcTemperature;
        ts = dt0 / 10.0;
    }
    // after an accepted step: true at the end, else on to the deepest pending one
    SSW_HD bool next(double dt0) {
        if (lo == 0 && hi == 0) return true;
        if (hi) {
            depth = 127 - __builtin_clzll(hi);
            hi &= ~(1ull << (depth - 64));
        } else {
            depth = 63 - __builtin_clzll(lo);
            lo &= ~(1ull << depth);
        }
        dt = dt0;
        for (int k = 0; k < depth; k++) dt = dt / 2.0;
        return false;
    }
    // after a rejected step: on to the first of its halves
    SSW_HD void halve() {
        depth += 1;
        if (depth < 64) lo |= 1ull << depth;
        else hi |= 1ull << (depth - 64);
        dt = dt / 2.0;
    }
};

// One attempt of perform_timestep (:394-441); true when the walk has ended,
// with its timescale in w.ts (dt0 / 10 and w.failed on depth overflow).
template <typename Ev>
SSW_HD bool walk_step(Cell& c, const Floor& f, double dt0, double safety, Walk& w, const Ev& ev) {
    clamp_state(c, f);
    double T0 = c.T, x0 = c.x;
    if (w.depth > kMaxDepth) {
        w.overflow(dt0);
        return true;
    }
    if (try_step(c, f, w.dt, safety, w.ts, w.proc, heat_rates(c, ev), ev)) return w.next(dt0);
    c.T = T0;
    c.x = x0;
    w.halve();
    return false;
}

// perform_timestep (:394-441). Returns the timescale; *failed on depth overflow.
SSW_HD double perform_timestep(Cell& c, const Floor& f, double dt0, double safety, int& proc, bool& failed) {
    Walk w;
    w.dt = dt0;
    while (!walk_step(c, f, dt0, safety, w, Serial())) {
    }
    proc = w.proc;
    failed = w.failed;
    return w.ts;
}

}  // namespace ssw
