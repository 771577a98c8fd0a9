// The field driver's first chord trial against the serial search: for random
// momenta, fields, directions and step lengths, every trial that
// first_chord_trial passes over must be one that the search shrinks by its
// full factor, and the trial it starts from the one that the search reaches.
//
// Usage: chord_trials count seed
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "field/FieldPropagator.hh"

using namespace celeritas_amd;

int main(int argc, char** argv)
{
    long const count = argc > 1 ? std::atol(argv[1]) : 100000;
    std::mt19937_64 gen(argc > 2 ? std::atol(argv[2]) : 1);
    std::uniform_real_distribution<double> u01(0, 1);
    auto log_uniform = [&](double lo, double hi) {
        return std::pow(10.0, lo + (hi - lo) * u01(gen));
    };
    FieldDriverOptions o;
    long skipped = 0, trials = 0, plain = 0, bad = 0;
    for (long i = 0; i < count; ++i)
    {
        o.delta_chord = log_uniform(-4, 0);
        o.max_nsteps = i % 5 == 0 ? 20 : 100;
        o.min_chord_shrink = i % 11 == 0 ? 0.3 : 0.5;
        double b[3], d[3];
        for (int k = 0; k < 3; ++k)
        {
            b[k] = 2 * u01(gen) - 1;
            d[k] = 2 * u01(gen) - 1;
        }
        if (i % 2 == 0)
        {
            b[0] = b[1] = 0;
            if (i % 6 == 0)  // nearly along the field
            {
                d[0] = log_uniform(-12, -1);
                d[1] = i % 12 == 0 ? 0 : log_uniform(-12, -1);
            }
            if (i % 42 == 0)
                d[0] = d[1] = 0;
        }
        double const bn = std::sqrt(field::dot3(b, b));
        double const dn = std::sqrt(field::dot3(d, d));
        double const tesla = log_uniform(-3, 1.5);
        double const p = log_uniform(-3, 6);
        field::UniformFieldStepper step;
        step.coeff = (i % 3 ? 1 : -1) * field::lorentz_per_cm_tesla;
        field::OdeState beg;
        for (int k = 0; k < 3; ++k)
        {
            step.b[k] = b[k] / bn * tesla;
            beg.pos[k] = 200 * u01(gen) - 100;
            beg.mom[k] = d[k] / dn * p;
        }
        double const h0 = i % 997 == 0 ? HUGE_VAL : log_uniform(-4, 24);
        field::ChordTrial const t = field::first_chord_trial(o, step, h0, beg.mom);
        // Serial search up to the same trial
        double h = h0;
        int remaining = o.max_nsteps;
        while (remaining > t.remaining)
        {
            field::StepperResult const r = step(h, beg);
            double const dchord = field::distance_chord(beg.pos, r.mid.pos, r.end.pos);
            if (!(dchord > o.delta_chord + o.dchord_tol)
                || std::sqrt(o.delta_chord / dchord) > o.min_chord_shrink)
                break;
            h *= o.min_chord_shrink;
            --remaining;
            ++skipped;
        }
        ++trials;
        plain += t.remaining == o.max_nsteps;
        if (remaining != t.remaining || !(h == t.step) || t.remaining < 1)
        {
            if (++bad < 10)
            {
                std::printf("draw %ld: p %g B %g h %g: starts at %g (%d left), search at "
                            "%g (%d left)\n",
                            i, p, tesla, h0, t.step, t.remaining, h, remaining);
            }
        }
    }
    std::printf("%ld searches, %ld from their first trial, %ld trials passed over, %ld differ\n",
                trials, plain, skipped, bad);
    return bad == 0 ? 0 : 1;
}
