// The tracker's short forms against the general ones, on params built by the
// library's host code:
// - is_behind of a conjunction (left at its first face with the other sense)
//   against the senses of all faces and the logic program, for every face of
//   every volume, both senses, points in the world and on the faces;
// - the safety distance of a plane normal to an axis against the distance to
//   the intersection along its normal.
//
// Usage: geo_rules problem.json points; prints the conjunctions, the
// comparisons and the differences.
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <random>
#include <sstream>

#include "geo/OrangeLiteTracker.hh"
#include "global/CoreParams.hh"

using namespace celeritas_amd;

int main(int argc, char** argv)
{
    if (argc != 3)
        return 2;
    std::ifstream f(argv[1]);
    std::stringstream ss;
    ss << f.rdbuf();
    auto params = CoreParams::from_json(ss.str());
    GeoParamsRef const& p = params->device_ref().geo;
    int const points = std::atoi(argv[2]);

    std::mt19937_64 rng(3);
    std::uniform_real_distribution<double> uniform(-1, 1);
    unsigned long conjunctions = 0, compared = 0, differ = 0;
    for (std::uint32_t v = 0; v < p.num_volumes; ++v)
    {
        VolumeRecord const record = p.volumes[v];
        conjunctions += (record.flags & conjunction) ? 1 : 0;
        double const* box = p.vol_bbox + 6 * v;
        for (int face = 0; face < record.num_faces; ++face)
        {
            SurfaceRecord const s = p.faces[record.face_begin + face];
            for (int i = 0; i < points; ++i)
            {
                // About the volume's box; every other point on the face
                double x[3];
                for (int k = 0; k < 3; ++k)
                {
                    bool const finite = std::isfinite(box[k]) && std::isfinite(box[3 + k]);
                    double const mid = finite ? 0.5 * (box[k] + box[3 + k]) : 0;
                    double const half = finite ? 0.5 * (box[3 + k] - box[k]) : 1000;
                    x[k] = mid + 1.1 * half * uniform(rng);
                }
                if (s.type <= SurfaceType::pz && i % 2)
                    x[static_cast<int>(s.type)] = s.coeff;
                for (bool sense : {false, true})
                {
                    int on;
                    std::uint32_t const mask = geo::calc_sense_mask(
                        p, v, x, geo::find_face(p, v, s.id), sense, &on);
                    bool const want = geo::eval_logic(p, v, mask);
                    ++compared;
                    differ += geo::is_behind(p, v, s.id, sense, x) != want ? 1 : 0;
                }
                if (s.type <= SurfaceType::pz)
                {
                    int const ax = static_cast<int>(s.type);
                    int const side = geo::calc_sense(p, s, x);
                    double n[3] = {0, 0, 0}, isect[2] = {0, 0};
                    n[ax] = side > 0 ? -1 : 1;
                    if (side != 0)
                        geo::calc_intersections(p, s, x, n, false, isect);
                    ++compared;
                    differ += geo::calc_safety_distance(p, s, x) != isect[0] ? 1 : 0;
                }
            }
        }
    }
    std::printf("%lu %lu %lu\n", conjunctions, compared, differ);
    return 0;
}
