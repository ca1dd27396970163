// gdp_arith.h - scalar propagation arithmetic shared by the HIP kernels and
// the host propagators of libGpuProp.so.
//
// The formulas are those of the reference's sequential propagator
// (src/propagation_methods.cuh:40-276, src/def.h:68-79) because the bounds the
// GPU returns must agree bit for bit with that propagator's arithmetic.  All
// operations are plain IEEE double operations evaluated one at a time (the
// library is compiled with -ffp-contract=off), division is the correctly
// rounded IEEE divide, and floor/ceil are exact, so host and device produce
// identical results from identical inputs.
#pragma once

#include <math.h>

#if defined(__HIPCC__)
#define GDP_HD __host__ __device__ __forceinline__
#else
#define GDP_HD static inline
#endif

namespace gdp {

constexpr double kInf = 1e20;
constexpr double kEps = 1e-9;
constexpr int kMaxRounds = 100;
constexpr int kVarContinuous = 3;

// Segment length of the canonical activity order: a row is summed segment by
// segment (pairwise tree over the entries of a segment in natural order,
// segment sums added left to right from +0.0).  A format constant shared by
// every kernel and the oracle.
constexpr int kSegLen = 256;

GDP_HD bool eps_le(double x, double y) { return (x - y) <= kEps; }
GDP_HD bool eps_lt(double x, double y) { return (x - y) < -kEps; }
GDP_HD bool eps_ge(double x, double y) { return (x - y) >= -kEps; }
GDP_HD bool eps_gt(double x, double y) { return (x - y) > kEps; }
// eps_ge(x, kInf) and eps_le(x, -kInf): doubles next to 1e20 lie 16384 apart,
// so the tolerance never decides and one comparison gives the same answer.
GDP_HD bool is_pos_inf(double x) { return x >= kInf; }
GDP_HD bool is_neg_inf(double x) { return x <= -kInf; }

// Storage class of a column from its bound envelope [l, u]: 0 = 2 x int16,
// 1 = 2 x int32, 2 = 2 x double.
GDP_HD int column_class(int vartype, double l, double u) {
    if (vartype == kVarContinuous) return 2;
    // both within the int32 range (false for NaN and infinities), then
    // integral: exact through a 64-bit integer round trip in that range,
    // without the library calls of floor()
    if (!(l >= -2147483647.0 && l <= 2147483647.0 && u >= -2147483647.0 && u <= 2147483647.0)) return 2;
    if (static_cast<double>(static_cast<long long>(l)) != l || static_cast<double>(static_cast<long long>(u)) != u)
        return 2;
    return l >= -32767.0 && l <= 32767.0 && u >= -32767.0 && u <= 32767.0 ? 0 : 1;
}
// An int16 column that needs 2 bits: its envelope lies in [0, 1].
GDP_HD bool binary_envelope(double l, double u) { return l >= 0.0 && u <= 1.0; }

// Contributions of a_k * x_k to the row's minimum and maximum activity and
// whether they are infinite (propagation_methods.cuh:198-213).  An infinite
// contribution is counted and contributes +0.0 to the finite part.
struct Contribution {
    double min_part, max_part, delta;
    int min_inf, max_inf;
};

GDP_HD Contribution contribution(double a, double l, double u) {
    Contribution c;
    const bool pos = a > kEps;  // eps_gt(a, 0)
    c.min_inf = pos ? is_neg_inf(l) : is_pos_inf(u);
    c.max_inf = pos ? is_pos_inf(u) : is_neg_inf(l);
    c.min_part = c.min_inf ? 0.0 : (a > 0 ? a * l : a * u);
    c.max_part = c.max_inf ? 0.0 : (a > 0 ? a * u : a * l);
    c.delta = fabs(a) * (u - l);
    return c;
}

// Row gate of the sequential propagator (propagation_methods.cuh:136-154):
// a row is skipped when no variable can move by more than the tolerance.
GDP_HD bool row_gate(double minact, double maxact, int min_inf, int max_inf,
                     double lhs, double rhs, double delta_max) {
    if (min_inf > 1 && max_inf > 1) return false;
    if (eps_lt(delta_max, kInf)) {
        const double a = rhs - minact, b = maxact - lhs;
        return !eps_le(delta_max, (b < a) ? b : a);
    }
    return true;
}

// Largest |a|(u-l) as the sequential propagator accumulates it: a later term
// replaces the running value only when larger by more than the tolerance
// (propagation_methods.cuh:198-201).
GDP_HD double eps_max_step(double running, double d) { return eps_gt(d, running) ? d : running; }

// Candidate bound of one variable from one side of a row
// (propagation_methods.cuh:40-52, :78-134): an upper bound v + l or a lower bound
// v + u, v the side's slack or surplus over the coefficient; `num_inf` is the
// infinity count of the activity it is derived from, and the other bound
// drops out when it is the one infinite contribution.  Lower bounds are
// computed mirrored (ceil(v - eps) = -floor(-v + eps); v = eps gives +0, whose
// sign only the accepted bounds need), so that both kinds share their
// instructions in a wave.  Returns whether it tightens.
GDP_HD bool candidate(bool upper, double v, int num_inf, double l, double u, bool is_cont, double &nb) {
    if (num_inf == 0) {
        v += upper ? l : u;
    } else if (num_inf != 1 || !(upper ? is_neg_inf(l) : is_pos_inf(u))) {
        return false;
    }
    const double x = upper ? v : -v;
    const double w = is_cont ? x : floor(x + kEps);
    if (!eps_lt(w, upper ? u : -l)) return false;
    nb = upper ? w : -w;
    if (!upper && !is_cont && x == -kEps) nb = 0.0;
    return true;
}

// New upper / lower bound from one row, `num_inf` the infinity count of the
// activity it is derived from.
GDP_HD bool tighten_upper(double a, double slack, double surplus, int num_inf,
                          double l, double u, bool is_cont, double &nb) {
    return candidate(true, (a > 0 ? slack : surplus) / a, num_inf, l, u, is_cont, nb);
}
GDP_HD bool tighten_lower(double a, double slack, double surplus, int num_inf,
                          double l, double u, bool is_cont, double &nb) {
    return candidate(false, (a > 0 ? surplus : slack) / a, num_inf, l, u, is_cont, nb);
}

// Both candidate bounds of one variable from one row, with the
// per-variable gates of propagation_methods.cuh:223-276.  Both candidates
// are computed from the same (l, u).  The right side bounds a positive
// coefficient's variable from above and any other's from below, the left
// side the other way round.  Returns bit 0 = lower tightened,
// bit 1 = upper tightened.
GDP_HD int tighten_variable(double a, double lhs, double rhs, double minact, double maxact,
                            int min_inf, int max_inf, bool is_cont, double l, double u,
                            double &nl, double &nu) {
    const bool pos = a > 0.0;
    const double width = pos ? a * (u - l) : a * (l - u);
    const double slack = rhs - minact;
    double nb;
    int r = 0;
    if (eps_gt(width, slack) && !is_pos_inf(rhs) && !is_neg_inf(minact) &&
        candidate(pos, slack / a, min_inf, l, u, is_cont, nb)) {
        if (pos) nu = nb;
        else nl = nb;
        r = pos ? 2 : 1;
    }
    if (eps_gt(width, maxact - lhs) && !is_neg_inf(lhs) && !is_pos_inf(maxact) &&
        candidate(!pos, (lhs - maxact) / a, max_inf, l, u, is_cont, nb)) {
        if (pos) nl = nb;
        else nu = nb;
        r |= pos ? 1 : 2;
    }
    return r;
}

// Whether the launch of double-buffered round `step` runs, as far as the unit's
// state says (`infeasible`: the round that crossed bounds, 0: none; `unusable`:
// crossed or outside the envelope as loaded).  The launch itself reports the
// crossings of round step - 1, so that value says nothing: waves that start
// late must decide as the first ones did, for the barriers of their workgroup.
// An earlier crossing is a smaller number.
GDP_HD bool round_runs(int step, int infeasible, bool unusable) {
    return !unusable && (infeasible == 0 || infeasible == step - 1);
}

}  // namespace gdp
