// Host-side check of the rule that picks the list build's form (nbuild_form):
// what is staged fits, the larger staging is used where only it fits, a forced
// staging is obeyed at every size, and several lanes per position (of which only
// one works where nothing is staged) only where the rows fit.  Prints one line
// per failure and "ok" at the end; exit status 1 on a failure.
#include "mdx_device.h"

#include <cmath>
#include <cstdio>

using namespace mdx;

static int fails = 0;

static void expect(bool c, const char *what, double n, double per_row)
{
    if (!c) {
        std::printf("FAIL %s n=%g per_row=%g\n", what, n, per_row);
        fails++;
    }
}

int main()
{
    const long long sizes[] = {1, 63, 64, 4096, 20000, 99999, 100000, 100001, 1 << 20, 1 << 27};
    const double per_row[] = {0.0, 1e-3, 0.5, 3, 41, 69, 110, 180, 200, 240, 259, 260, 400, 2000};
    for (long long n : sizes)
        for (double r : per_row) {
            const double held = r > 0 ? (std::ceil(64 / r) + 3) * r : 0;
            const NbForm f = nbuild_form(n, r, -1);
            const bool staged = held <= 0.9 * NB_CAP_D;
            expect(f.lanes == (n <= 100000 && staged ? 4 : 1), "four lanes where staged", n, r);
            if (f.lanes == 4)
                expect(f.dense == !(held <= 0.9 * NB_CAP_S), "larger where only it fits", n, r);
            expect(nbuild_form(n, r, 1).dense == 1, "forced larger", n, r);
            expect(nbuild_form(n, r, 0).dense == 0, "forced smaller", n, r);
        }
    // the sizes the forms were measured at
    expect(nbuild_form(4096, 16, -1).lanes == 4, "4,096 fluid", 4096, 16);
    expect(nbuild_form(1 << 20, 68, -1).dense == 0, "1M condensate", 1 << 20, 68);
    std::puts(fails ? "failed" : "ok");
    return fails != 0;
}
