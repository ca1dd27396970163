// The decision of a round's launch to run (gdp_arith.h, round_runs): every
// wave of the launch takes the same one, whether it starts before or after
// another wave of the launch has reported a crossing of the round before.
// Prints "ok" and exits 0.
#include <cstdio>

#include "gdp_arith.h"

int main() {
    for (int step = 1; step <= gdp::kMaxRounds; step++) {
        const int own = step - 1;  // what this launch writes (round 1 looks for no crossing)
        bool ok = gdp::round_runs(step, 0, false) && gdp::round_runs(step, own, false);
        ok &= !gdp::round_runs(step, 0, true) && !gdp::round_runs(step, own, true);
        for (int earlier = 1; earlier < own; earlier++) ok &= !gdp::round_runs(step, earlier, false);
        if (!ok) {
            std::printf("round %d\n", step);
            return 1;
        }
    }
    std::printf("ok\n");
    return 0;
}
