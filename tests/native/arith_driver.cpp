// Candidate bounds of gdp_arith.h against the formulas they come from
// (propagation_methods.cuh:40-52, :78-134: floor(v + eps) for upper, ceil(v -
// eps) for lower bounds of integer columns), bit for bit, zeros' signs
// included, over all pairs of values around the tolerance, integers, halves,
// the infinities of the encoding and beyond.  Prints "ok" and exits 0.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "gdp_arith.h"

static bool direct(bool upper, double v, int num_inf, double l, double u, bool cont, double &nb) {
    if (num_inf == 0) v += upper ? l : u;
    else if (num_inf != 1 || !(upper ? gdp::is_neg_inf(l) : gdp::is_pos_inf(u))) return false;
    if (upper) {
        v = cont ? v : std::floor(v + gdp::kEps);
        if (!(v - u < -gdp::kEps)) return false;
    } else {
        v = cont ? v : std::ceil(v - gdp::kEps);
        if (!(v - l > gdp::kEps)) return false;
    }
    nb = v;
    return true;
}

int main() {
    std::vector<double> vals;
    for (double x : {0.0, 1e-9, 0.5e-9, 2e-9, 1e-300, 0.3, 0.5, 1.0, 1.0 + 1e-9, 1.0 - 1e-9, 2.5, 7.0, 32768.0, 2147483648.0,
                     9e15, 1e20, 1e300, HUGE_VAL})
        for (double s : {1.0, -1.0})
            for (double y : {x, std::nextafter(x, 1e308), std::nextafter(x, -1e308)}) vals.push_back(s * y);
    for (double v : vals)
        for (double l : vals)
            for (double u : vals)
                for (int k = 0; k < 12; k++) {
                    const bool upper = k & 1, cont = k & 2;
                    const int inf = k >> 2;
                    double a = 42.0, b = 42.0;
                    const bool ra = direct(upper, v, inf, l, u, cont, a);
                    const bool rb = gdp::candidate(upper, v, inf, l, u, cont, b);
                    if (ra != rb || std::memcmp(&a, &b, sizeof(a)) != 0) {
                        std::printf("%s v=%a l=%a u=%a inf=%d cont=%d: %d %a, want %d %a\n", upper ? "upper" : "lower", v,
                                    l, u, inf, cont, rb, b, ra, a);
                        return 1;
                    }
                }
    std::printf("ok\n");
    return 0;
}
