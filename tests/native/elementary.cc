// Largest errors of the FP64 logarithm, sine and cosine against the extended
// type of the host, in units of the last place, over a named range.
//
//   elementary <log|sin|cos> <low> <high> <count>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>

#include "corecel/Elementary.hh"

using namespace celeritas_amd;

int main(int argc, char** argv)
{
    if (argc < 5)
        return 2;
    std::string const fn = argv[1];
    double const lo = std::atof(argv[2]), hi = std::atof(argv[3]);
    int const count = std::atoi(argv[4]);
    std::mt19937_64 rng(5);
    std::uniform_real_distribution<double> uniform(0, 1);
    double worst = 0, at = 0;
    for (int i = 0; i < count; ++i)
    {
        // A positive range over decades is sampled by its logarithm
        double const u = uniform(rng);
        long double const ratio = static_cast<long double>(hi) / lo;
        double const x = (lo > 0 && ratio > 1e3) ? static_cast<double>(lo * powl(ratio, u))
                                                 : lo + (hi - lo) * u;
        double s, c, got;
        long double want;
        if (fn == "log")
        {
            got = elem::log(x);
            want = logl(x);
        }
        else
        {
            elem::sincos(x, &s, &c);
            got = fn == "sin" ? s : c;
            want = fn == "sin" ? sinl(x) : cosl(x);
        }
        if (want == 0)
            continue;
        int e;
        std::frexp(static_cast<double>(want), &e);
        double const err = std::fabs(static_cast<double>((got - want) / ldexpl(1.0L, e - 53)));
        if (!(err <= worst))
        {
            worst = err;
            at = x;
        }
    }
    double const inf = HUGE_VAL;
    bool const special = elem::log(0.0) == -inf && elem::log(-0.0) == -inf
                         && elem::log(inf) == inf && std::isnan(elem::log(-1.0))
                         && std::isnan(elem::log(-inf)) && std::isnan(elem::log(std::nan("")))
                         && elem::log(1.0) == 0 && elem::sin(0.0) == 0
                         && elem::cos(0.0) == 1 && std::isnan(elem::sin(std::nan("")));
    std::printf("%.4f %.17g %d\n", worst, at, special ? 1 : 0);
    return 0;
}
