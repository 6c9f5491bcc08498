// trav_pack_host.cpp -- test infrastructure: the traversal's node packing
// (bisemutum-engine_amd/csrc/pt_trav.hpp) as a CPU library, for comparison with the nodes a
// GPU build has made.
#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../bisemutum-engine_amd/csrc/pt_trav.hpp"

// n nodes: child[4 k + j] links (0: empty), box[24 k + 4 a + j] coordinate a (lo xyz, hi xyz)
// of child j's exact box; out: n x 64 B.
extern "C" void trav_pack_nodes(int64_t n, const int32_t* child, const float* box, void* out) {
    for (int64_t k = 0; k < n; ++k) {
        float b[4][6];
        int cnt = 0;
        while (cnt < 4 && child[4 * k + cnt] != 0) ++cnt;
        for (int j = 0; j < 4; ++j)
            for (int a = 0; a < 6; ++a) b[j][a] = box[24 * k + 4 * a + j];
        const bipt::TravNode r = bipt::trav_pack(b, child + 4 * k, cnt);
        std::memcpy(static_cast<char*>(out) + 64 * k, &r, 64);
    }
}
