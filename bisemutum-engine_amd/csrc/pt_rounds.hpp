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
// server): all configured ones, unless the call itself is so small that the tree is likely
// a preview's (a round costs ~0.1-0.5 ms).
inline uint32_t kept_rounds(uint64_t paths, uint32_t tris, uint32_t configured) {
    return paths >= std::max<uint64_t>(4ull * tris, 1ull << 20) ? configured : 0u;
}

// Rounds that a call's own paths repay, at most `configured`: for trees that no later call
// traces.  Round k runs when the call traces at least (2^21 + 32 n) (1 + k (k - 1) / 3) paths
// of the scene's n triangles (paths of fewer than four segments count in proportion): the
// first round saves most, the third a tenth of it, and each costs the same.  Frame with
// 0 / 1 / 2 / 3 rounds, build included:
//   atrium (262k), 8 segments, 2.1 M paths   5.52 /  5.55 /  5.85 /  6.21 ms
//                              4.1 M         8.88 /  8.40 /  8.62 /  8.91
//                             16.6 M        28.68 / 25.21 / 24.91 / 25.10
//                             33.2 M        55.2  / 47.7  / 46.8  / 46.6
//   rooms of 20k, 6 segments,  1.8 M         3.01 /  3.05 /  3.27 /  3.49
//                              7.4 M         7.49 /  7.03 /  7.14 /  7.32
//   250k                       7.4 M         6.86 /  7.08 /  7.64 /  8.11
//   900k                       8.3 M        11.31 / 13.34 / 14.85 / 16.38
inline uint32_t paid_rounds(uint64_t full_paths, uint32_t tris, uint32_t configured) {
    const uint64_t first = (1ull << 21) + 32ull * tris;
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
