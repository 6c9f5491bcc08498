// pt_rounds.hpp -- how many treelet rounds a render's LBVH build runs (host only; plain
// C++, so that tests compile it without a GPU).
#pragma once

#include <stdint.h>

#include <algorithm>

namespace bipt {

// What a scene's context has seen of the use of its trees.
struct TreeUse {
    bool rendered = false;   // a render has built a tree of the present scene
    bool outlived = false;   // a tree has been traced, or asked to be kept, beyond the call that built it
};

// Rounds of a tree that later calls trace too (renders that keep it, ray queries, the
// server): all configured ones, unless the call itself is so small that the tree is likely a
// preview's (a round costs 0.2 ms for 20k triangles, 0.4 to 0.8 ms for 260k, 1.4 to 3 ms for 900k).
inline uint32_t kept_rounds(uint64_t paths, uint32_t tris, uint32_t configured) {
    return paths >= std::max<uint64_t>(4ull * tris, 1ull << 20) ? configured : 0u;
}

// Rounds that a call's own paths repay, at most `configured`: for trees that no later call
// traces.  Round k runs when the call traces at least (2^21 + 20 n) (1 + k (k - 1) / 3) paths
// of the scene's n triangles (paths of fewer than four segments count in proportion): the
// first round saves most, the third a tenth of it, and each costs the same.  Frame with
// 0 / 1 / 2 / 3 rounds, build included, ms:
//   atrium (262k), 8 segments, 2.1 M paths   4.97 /  4.97 /  5.26 /  5.60
//                              4.1 M         8.15 /  7.66 /  7.89 /  8.17
//                              8.3 M        14.55 / 13.16 / 13.21 / 13.43
//                             16.6 M        27.17 / 23.87 / 23.58 / 23.66
//                             33.2 M        52.58 / 45.43 / 44.49 / 44.29
//   rooms of 20k, 6 segments,  1.8 M         2.75 /  2.78 /  2.99 /  3.20
//                              3.7 M         4.13 /  4.01 /  4.20 /  4.39
//                              7.4 M         6.88 /  6.42 /  6.57 /  6.73
//   100k                       3.7 M         3.27 /  3.41 /  3.73 /  4.00
//                              7.4 M         5.10 /  5.05 /  5.33 /  5.61
//                             16.6 M         9.56 /  9.09 /  9.31 /  9.60
//   250k                       7.4 M         6.75 /  6.91 /  7.49 /  7.94
//                             16.6 M        16.34 / 15.28 / 15.69 / 16.14
//   900k                       7.4 M         8.23 / 10.47 / 12.27 / 13.72
//                             16.6 M        16.44 / 17.64 / 19.16 / 20.83
// A path of the atrium saves about twice what a room's does, so the line lies between: at
// 32 n the atrium's 8.3 M paths went without (8% slower than three rounds), below 16 n the
// 900k room's 16.6 M got one (7% slower than none).
inline uint32_t paid_rounds(uint64_t full_paths, uint32_t tris, uint32_t configured) {
    const uint64_t first = (1ull << 21) + 20ull * tris;
    uint32_t k = 0;
    while (k < configured && 3ull * full_paths >= first * (3ull + (uint64_t)k * (k + 1ull))) ++k;
    return k;
}

// A call cannot know whether its tree will be traced again, so it goes by what it is told
// (`reuse`: the call keeps trees) and by what the context has seen: the first tree of a
// scene, and every tree of a context whose trees have been traced beyond their own call, gets
// the kept tree's rounds; a context that rebuilds call after call, with nothing in
// between, builds what each call repays.
inline uint32_t build_rounds(const TreeUse& use, bool reuse, uint64_t paths, uint64_t full_paths, uint32_t tris,
                             uint32_t configured) {
    if (reuse || use.outlived || !use.rendered) return kept_rounds(paths, tris, configured);
    return paid_rounds(full_paths, tris, configured);
}

}  // namespace bipt
