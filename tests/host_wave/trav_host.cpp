// trav_host.cpp -- test infrastructure: the traversal's node packing and visit test
// (bisemutum-engine_amd/csrc/pt_trav.hpp) compiled for the CPU and compared with the exact
// FP32 slab test, box by box and ray by ray.  Reads records of (4 boxes, child count, ray
// origin, direction, extent) and prints, over all of them, how many boxes the exact test
// passes, how many of those the visit test skips (must be none), and how many it visits.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../bisemutum-engine_amd/csrc/pt_trav.hpp"

using namespace bipt;

static float safe_inv(float x) {   // trace.hip
    float ax = x < 0.0f ? -x : x;
    if (ax < 1e-20f) x = x < 0.0f ? -1e-20f : 1e-20f;
    return 1.0f / x;
}

// The exact test of trace.hip (box_exact) and of the CPU restatement.
static bool exact(const float* b, const float* o, const float* inv, float tmin, float tmax) {
    float n[3], f[3];
    for (int a = 0; a < 3; ++a) {
        const float t0 = (b[a] - o[a]) * inv[a], t1 = (b[3 + a] - o[a]) * inv[a];
        n[a] = std::fmin(t0, t1);
        f[a] = std::fmax(t0, t1);
    }
    const float tn = std::fmax(std::fmax(n[0], n[1]), std::fmax(n[2], tmin));
    const float tf = std::fmin(std::fmin(f[0], f[1]), std::fmin(f[2], tmax));
    return tn <= tf * 1.00000036f;
}

struct Rec {
    float box[4][6];
    int32_t n;
    float o[3], d[3], tmax;
};

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    FILE* f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    Rec r;
    long total = 0, hit = 0, skipped = 0, visited = 0, order = 0;
    while (std::fread(&r, sizeof r, 1, f) == 1) {
        const int32_t id[4] = {1, ~0, 2, ~1};
        const TravNode nd = trav_pack(r.box, id, r.n);
        TravRay ray;
        float inv[3];
        for (int a = 0; a < 3; ++a) {
            inv[a] = safe_inv(r.d[a]);
            trav_ray_axis(ray, a, r.o[a], inv[a]);
        }
        TravPlanes p;
        for (int a = 0; a < 3; ++a)
            trav_planes_axis(p, a, ray, nd.base[a], nd.scale[a], nd.plane[2 * a], nd.plane[2 * a + 1]);
        for (int k = 0; k < 4; ++k) {
            if (k >= r.n) {
                if (nd.child[k] != 0) return 3;
                continue;
            }
            if (nd.child[k] != id[k]) return 3;
            float tn;
            const bool v = trav_visit(p, k, r.tmax, &tn), e = exact(r.box[k], r.o, inv, 0.001f, r.tmax);
            ++total;
            hit += e;
            visited += v;
            skipped += e && !v;
            order += v && !(tn >= 0.0f);   // the entry distance orders children: a number
        }
    }
    std::fclose(f);
    std::printf("%ld %ld %ld %ld %ld\n", total, hit, skipped, visited, order);
    return 0;
}
