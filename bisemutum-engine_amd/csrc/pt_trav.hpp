// pt_trav.hpp -- the traversal's node record and its visit test (host and device; plain
// C++, so that tests compile it for the CPU).
//
// The box test of a node only decides which nodes a ray visits; whether a leaf's hit counts
// is decided by the exact FP32 slab test of the leaf's own box (trace.hip).  So a node need
// not hold exact boxes: it may visit too much, never too little.  With the 128-B node of
// FP32 planes (seven 16-B loads per visited node) the traversal kernels were bound by the
// rate of those loads -- a CU's vector cache takes about one lane's 16-B line per clock when
// every lane reads its own node: 38 busy lanes x 7 loads = 266 clocks a step and wavefront,
// more than the arithmetic takes.  This record takes four loads, half the bytes, and 24
// more conversions.  Atrium, 16 spp at 1080p: closest hit 21.5 -> 19.9 ms and shadow rays
// 15.3 -> 12.8 ms per frame from the record alone.
//
// A node's four child boxes are stored as 8-bit planes in the node's own frame: plane q of
// axis a stands at base[a] + q * scale[a].  Low planes are rounded down and high planes up, by
// at least kTravSlack quanta each unless they lie at the frame's own edge (q = 0), which the
// rounding errors of the visit test below need.  An axis with a coordinate beyond 1e18
// (whose product with an inverse direction of up to 1e20 could overflow) or one that is no
// number gets scale = +inf and q = 0: the visit test's products are then NaN, which fminf
// and fmaxf ignore, so the axis rejects nothing.  An empty slot has link 0, the root's index, which is no node's child.
#pragma once

#include <stdint.h>

#ifndef PT_HD
#ifdef __HIPCC__
#define PT_HD __host__ __device__ __forceinline__
#else
#define PT_HD inline
#endif
#endif

namespace bipt {

struct alignas(64) TravNode {
    float base[3], scale[3];
    uint32_t plane[6];  // byte k: child k's planes (low x, high x, low y, high y, low z, high z)
    int32_t child[4];   // internal: node index > 0; leaf j: ~j; empty slot: 0
};
static_assert(sizeof(TravNode) == 64, "traversal node is 64 bytes");

constexpr float kTravSlack = 0.0625f;

// Frame of one axis for used boxes [lo, hi] (n of them); returns false for an axis that
// rejects nothing.
PT_HD bool trav_frame(const float* lo, const float* hi, int n, float* base, float* scale) {
    float l = lo[0], h = hi[0];
    bool fine = true;
    for (int k = 0; k < n; ++k) {
        fine = fine && lo[k] >= -1e18f && hi[k] <= 1e18f && lo[k] <= hi[k];   // false for NaN
        l = lo[k] < l ? lo[k] : l;
        h = hi[k] > h ? hi[k] : h;
    }
    if (!fine) {
        *base = 0.0f;
        *scale = __builtin_inff();
        return false;
    }
    // 252 quanta for the extent, one for each edge, the rest for rounding; never zero
    float s = (h - l) * (1.0f / 252.0f) * 1.000001f;
    s = s < 0x1p-100f ? 0x1p-100f : s;
    *scale = s;
    *base = l - s;
    return true;
}
PT_HD uint32_t trav_lo(float x, float base, float scale) {
    const float q = __builtin_floorf((x - base) / scale - kTravSlack);
    return q <= 0.0f ? 0u : q >= 255.0f ? 255u : (uint32_t)q;
}
PT_HD uint32_t trav_hi(float x, float base, float scale) {
    const float q = __builtin_ceilf((x - base) / scale + kTravSlack);
    return q >= 255.0f ? 255u : q <= 0.0f ? 0u : (uint32_t)q;
}
// The node of n children: box[k] = lo xyz, hi xyz; id[k] the links.
PT_HD TravNode trav_pack(const float (*box)[6], const int32_t* id, int n) {
    TravNode r;
    for (int a = 0; a < 3; ++a) {
        float lo[4], hi[4];
        for (int k = 0; k < 4; ++k) {
            lo[k] = box[k < n ? k : 0][a];
            hi[k] = box[k < n ? k : 0][3 + a];
        }
        const bool fine = trav_frame(lo, hi, n, &r.base[a], &r.scale[a]);
        uint32_t wl = 0u, wh = 0u;
        for (int k = 0; k < 4; ++k) {
            const uint32_t ql = k < n && fine ? trav_lo(lo[k], r.base[a], r.scale[a]) : 0u;
            const uint32_t qh = k < n && fine ? trav_hi(hi[k], r.base[a], r.scale[a]) : 0u;
            wl |= ql << (8 * k);
            wh |= qh << (8 * k);
        }
        r.plane[2 * a] = wl;
        r.plane[2 * a + 1] = wh;
    }
    for (int k = 0; k < 4; ++k) r.child[k] = k < n ? id[k] : 0;
    return r;
}

// The children of the traversal node made at node k of a BVH2 (whose nodes hold two child
// links and boxes, lo xyz and hi xyz): k's children, of which the internal one with the largest
// surface is replaced by its own two until there are four or only leaves.  Returns how many;
// id: links, box: exact boxes.
template <class Node>
PT_HD int trav_children(const Node* nodes, int k, int32_t (&id)[4], float (&box)[4][6]) {
    int cnt = 2;
    for (int c = 0; c < 2; ++c) {
        id[c] = nodes[k].child[c];
        for (int a = 0; a < 6; ++a) box[c][a] = nodes[k].box[6 * c + a];
    }
    while (cnt < 4) {
        int pick = -1;
        float best = -1.0f;
        for (int j = 0; j < cnt; ++j) {
            if (id[j] < 0) continue;
            const float dx = box[j][3] - box[j][0], dy = box[j][4] - box[j][1], dz = box[j][5] - box[j][2];
            const float half = (dx * dy + dy * dz) + dz * dx;
            if (half > best) { best = half; pick = j; }
        }
        if (pick < 0) break;
        const Node& m = nodes[id[pick]];
        id[cnt] = m.child[1];
        for (int a = 0; a < 6; ++a) box[cnt][a] = m.box[6 + a];
        id[pick] = m.child[0];
        for (int a = 0; a < 6; ++a) box[pick][a] = m.box[a];
        ++cnt;
    }
    return cnt;
}

// A ray as the visit test reads it: inverse direction, and per axis -(o inv) -/+ 4u |o inv|
// (u = 2^-24) for the planes met first and last.
//
// Where o inv overflows, |o| is above 3.4e18 (|inv| is at most 1e20), so every plane of a
// framed axis (|p| <= 1.004e18) lies at |(p - o) inv| >= 2.3e38, behind the ray or beyond any
// extent (at most 1.7e38): cn and cf are then the same infinity, which rejects the node as
// the exact test does.  (Left unconstrained, one ray with an infinite origin walks the whole
// tree.)  The same holds where o inv is finite and a sum below overflows.  An axis whose
// o inv is no number rejects nothing, as in the exact test.
struct TravRay {
    float inv[3], cn[3], cf[3];
};
PT_HD void trav_ray_axis(TravRay& r, int a, float o, float inv) {
    const float oi = o * inv, m = __builtin_fabsf(oi);
    const float slack = m <= 3.402823466e38f ? m * 0x1p-22f : 0.0f;   // none for an infinity (inf - inf)
    const bool number = oi == oi;
    r.inv[a] = inv;
    r.cn[a] = number ? -oi - slack : -__builtin_inff();
    r.cf[a] = number ? -oi + slack : __builtin_inff();
}

// One node as one ray sees it.  A plane q is met at
//   fma(q, scale inv, fma(base, inv, cn or cf)),
// the plane met first being the low one where inv is positive and the high one where it is
// negative: words of near and far planes are swapped once per axis and node instead of
// taking a minimum and a maximum per child.
//
// Why no box that the exact test passes is skipped: let p be a stored plane and
// r = (p - o) inv.  The rounding errors of the chain sum to at most
// 2.1u |o inv| + 2.1u |r| + 2.1u |q scale inv|.  The first is covered by the 4u |o inv| in cn and
// cf, the last (under 3.3e-5 quanta) by kTravSlack, and is zero for q = 0.  The exact test
// (fl(fl(p - o) inv), robust factor 1 + 6u) passes only boxes with
// r_near <= r_far (1 + 11.2u), so near <= far (1 + 16u); kTravVisit is 1 + 32u.  The clamp at the
// ray's start (kTravTMin) has the same room.  Distances at or behind the origin need no
// care: such a far plane fails both tests.
constexpr float kTravVisit = 1.0000019073486328125f;   // 1 + 2^-19
constexpr float kTravTMin = 0.00099999f;               // below the rays' start, 0.001
struct TravPlanes {
    float b[3], an[3], af[3];
    uint32_t nearq[3], farq[3];
};
PT_HD void trav_planes_axis(TravPlanes& p, int a, const TravRay& r, float base, float scale, uint32_t lo, uint32_t hi) {
    p.b[a] = scale * r.inv[a];
    p.an[a] = __builtin_fmaf(base, r.inv[a], r.cn[a]);
    p.af[a] = __builtin_fmaf(base, r.inv[a], r.cf[a]);
    const bool back = r.inv[a] < 0.0f;
    p.nearq[a] = back ? hi : lo;
    p.farq[a] = back ? lo : hi;
}
// Whether a ray of extent tmax visits child k; *tn: where it enters the box.
PT_HD bool trav_visit(const TravPlanes& p, int k, float tmax, float* tn) {
    float n[3], f[3];
    for (int a = 0; a < 3; ++a) {
        n[a] = __builtin_fmaf((float)((p.nearq[a] >> (8 * k)) & 255u), p.b[a], p.an[a]);
        f[a] = __builtin_fmaf((float)((p.farq[a] >> (8 * k)) & 255u), p.b[a], p.af[a]);
    }
    const float t0 = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(n[0], n[1]), n[2]), kTravTMin);
    const float t1 = __builtin_fminf(__builtin_fminf(__builtin_fminf(f[0], f[1]), f[2]), tmax);
    *tn = t0;
    return t0 <= t1 * kTravVisit;
}

}  // namespace bipt
