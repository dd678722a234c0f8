// Host-side check of PlaneFilter (pp_search.h): no target that plane_hit reports
// as hit may be passed over, whatever the rounding of the device's reciprocal
// (its 1 ulp either way). Built by tests/test_plane_filter_host.py.
//   usage: plane_check <scale> <seed> <n>   prints: hits passed_over let_through
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include <cstring>

#include "../../photonpropagation.jl_amd/csrc/pp_search.h"

using namespace pp;

int main(int argc, char** argv) {
    if (argc < 4) return 2;
    const float scale = (float)atof(argv[1]);
    std::mt19937_64 rng((unsigned)atoi(argv[2]));
    std::uniform_real_distribution<float> U(0.0f, 1.0f);
    std::normal_distribution<float> N(0.0f, 1.0f);
    long hits = 0, over = 0, through = 0;
    const long n = atol(argv[3]);
    for (long k = 0; k < n; ++k) {
        float d[3] = {N(rng), N(rng), N(rng)};
        const float special[] = {0.0f, -0.0f, 1e-40f, -1e-30f, 1e-7f, FLT_MIN};
        if (k % 7 == 0) d[2] = special[(k / 7) % 6];
        const float l = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const f3 dir = make3(d[0] / l, d[1] / l, d[2] / l);
        const f3 pos = make3(scale * N(rng), scale * N(rng), scale * N(rng));
        float step = k % 11 == 0 ? 0.0f : scale * -std::log(U(rng) + 1e-8f);
        const uint32_t kind = k & 1 ? PP_SHAPE_RECTANGLE : PP_SHAPE_DISC;
        const float a = scale * (0.01f + U(rng)), b = kind == PP_SHAPE_DISC ? a : scale * (0.01f + U(rng));
        // a target that the segment crosses near an edge of the shape or of the step
        float t = step * (k % 5 == 0 ? 1.0f : k % 5 == 1 ? 0.0f : U(rng));
        const float ux = k % 3 == 0 ? 1.0f : 2.0f * U(rng) - 1.0f, uy = 2.0f * U(rng) - 1.0f;
        const float4 tg = make_float4(pos.x + t * dir.x - ux * a, pos.y + t * dir.y - uy * b,
                                      pos.z + t * dir.z, kind == PP_SHAPE_DISC ? a * a : 0.0f);
        const float4 e = make_float4(0.0f, a, b, 0.0f);
        float dist;
        const bool hit = plane_hit(kind, tg, e, pos, dir, step, dist);
        PlaneFilter f(pos, dir, step);
        const float inv = f.inv_z;
        for (int u = -1; u <= 1; ++u) {
            f.inv_z = u < 0 ? std::nextafterf(inv, -INFINITY) : u > 0 ? std::nextafterf(inv, INFINITY) : inv;
            const bool miss = f.misses(tg, e, pos, dir);
            over += hit && miss;
            through += !hit && !miss;
        }
        hits += hit;
    }
    printf("%ld %ld %ld\n", hits, over, through);
    return 0;
}
