// Bytes of LDS that the step kernels' launches stage, from params built by
// the library's host code.
//
// Usage: staging problem.json; prints the regions (physics, distances, all
// geometry) and what is staged: physics alone (pre-step, interactions),
// distances (neutral along-step), all geometry (boundary), and physics and
// distances (charged along-step).
#include <cstdio>
#include <fstream>
#include <sstream>

#include "global/CoreParams.hh"
#include "global/StagingRules.hh"

using namespace celeritas_amd;

int main(int argc, char** argv)
{
    if (argc != 2)
        return 2;
    std::ifstream f(argv[1]);
    std::stringstream ss;
    ss << f.rdbuf();
    auto params = CoreParams::from_json(ss.str());
    CoreParamsRef const& p = params->device_ref();
    std::printf("%u %u %u %u %u %u %u\n", p.phys.hot_bytes, p.geo.track_bytes, p.geo.hot_bytes,
                staged_table_bytes(p), staged_geo_bytes(p), staged_crossing_bytes(p),
                staged_both_bytes(p));
    return 0;
}
