// trace.hip -- software BVH traversal on gfx950 (CDNA4 has no ray-tracing units).
//
// Replaces TraceRay of rt_gbuffer.hlsl:25 (closest hit, TMin 0.001, TMax
// ray_length) and the shadow-map lookups of lights.hlsl:69-101 (exact any-hit
// shadow rays).  Rays come from SoA queues (coalesced); the traversal structure is
// the BVH4 collapsed from the LBVH, one 64-B node per step (4 x 16-B loads, child boxes
// as 8-bit planes: pt_trav.hpp).  Node boxes only steer the traversal; a hit counts if the
// exact FP32 tests of its triangle and of its triangle's own box pass.  Short stack: the
// bottom `L` entries live in LDS ([slot][lane], bank conflict free for equal depths), deeper
// entries in a per-lane private array; the total depth bound kStackMax covers any tree
// the build can produce.
//
// Persistent lanes with dynamic ray fetch: a workgroup-resident grid of wavefronts
// keeps lanes busy -- lanes whose rays have finished take the next ray indices from
// per-XCD counters (one atomic per wavefront and refill, lanes ranked by a ballot), so
// secondary rays of very different lengths do not idle the SIMD.  Each step is
// node-centric: the four child boxes of one node are tested, hit leaves queued, the
// nearest hit internal child entered and the other hit internal children pushed
// (ascending slot order).
//
// What bounds it (atrium, 16 spp at 1080p, depth 8, SQ and TCP counters): VALU issue first, the
// vector cache close behind.  Extension rays issue 1.02 VALU instructions per clock and CU and
// look up 0.88 cache lines per clock and CU in the vector cache, whose limit is about one
// (shadow rays 0.85 and 0.79); with 128-B nodes of FP32 planes it was the lookups (seven 16-B
// loads a node).  Closest hit 24.4 -> 17.5 ms, shadow 16.5 -> 12.9 ms per frame from 64-B
// nodes (4 loads), near and far planes by the ray's signs and fused multiply-adds, winners'
// barycentrics kept in LDS instead of a second triangle test, and a step whose masks stay in
// scalar registers; per extension ray 94 -> 78 wavefront VALU instructions.
#include <algorithm>

#include "pt_kernels.hpp"

namespace bipt {
namespace {

// What a lane does, in one register: the node it visits next (>= 0), or
constexpr int kParked = -1;   // no node left: waits for its queued leaves to be tested
constexpr int kIdle = -2;     // no ray
constexpr uint32_t kNoRay = 0xffffffffu;

__device__ __forceinline__ V3 safe_inv(V3 d) {
    auto one = [](float x) {
        float ax = x < 0.0f ? -x : x;
        if (ax < 1e-20f) x = x < 0.0f ? -1e-20f : 1e-20f;
        return 1.0f / x;
    };
    return v3(one(d.x), one(d.y), one(d.z));
}

// Node and leaf records are read through global-address-space pointers (the integer
// round trip keeps the compiler from folding the cast away): global loads, not flat ones,
// so the 16-B loads of a node issue back to back and the waits count only vector
// memory (flat loads, which might address LDS, made the compiler wait between them).
typedef float VF4 __attribute__((ext_vector_type(4)));
typedef int VI4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const VF4 GlobalF4;
typedef __attribute__((address_space(1))) const char GlobalChar;

__device__ __forceinline__ TravRay trav_ray(V3 o, V3 d) {
    const V3 inv = safe_inv(d);
    TravRay r;
    trav_ray_axis(r, 0, o.x, inv.x);
    trav_ray_axis(r, 1, o.y, inv.y);
    trav_ray_axis(r, 2, o.z, inv.z);
    return r;
}

// A node's record in registers.
struct NodeRegs {
    VF4 n0, n1, n2;
    VI4 ch;
};
// SMALL: the nodes lie within 4 GB of `nodes`, which is the same for every lane (scalar
// base, 32-bit offset).
template <bool SMALL>
__device__ __forceinline__ void load_node(NodeRegs& r, const TravNode* nodes, int i) {
    GlobalChar* at = (GlobalChar*)(uintptr_t)nodes;
    if constexpr (SMALL) at += (uint32_t)i << 6;
    else at += (size_t)(uint32_t)i * sizeof(TravNode);
    GlobalF4* p = (GlobalF4*)at;
    r.n0 = p[0];
    r.n1 = p[1];
    r.n2 = p[2];
    r.ch = __builtin_bit_cast(VI4, p[3]);
}
__device__ __forceinline__ TravPlanes node_planes(const NodeRegs& n, const TravRay& r) {
    TravPlanes p;
    trav_planes_axis(p, 0, r, n.n0[0], n.n0[3], __float_as_uint(n.n1[2]), __float_as_uint(n.n1[3]));
    trav_planes_axis(p, 1, r, n.n0[1], n.n1[0], __float_as_uint(n.n2[0]), __float_as_uint(n.n2[1]));
    trav_planes_axis(p, 2, r, n.n0[2], n.n1[1], __float_as_uint(n.n2[2]), __float_as_uint(n.n2[3]));
    return p;
}

// Leaf intersection record held in registers: v0, e1, e2, the flag word, the low corner of
// the box (x, y); the rest of the box is read only where the triangle is hit.
struct LeafRegs {
    VF4 g0, g1, g2;
};
__device__ __forceinline__ LeafRegs load_leaf(const LeafGeo* geo, uint32_t leaf) {
    GlobalF4* p = (GlobalF4*)(uintptr_t)(geo + leaf);
    return LeafRegs{p[0], p[1], p[2]};
}
// The exact slab test of the leaf's own box for a ray extent up to tmax, as the CPU
// restatement computes it.  No operand can be NaN for a finite ray ((b - o) and inv are
// finite, inv nonzero), so fminf/fmaxf select what its comparisons select, up to the sign
// of zero, which only ever reaches comparisons.
__device__ __forceinline__ bool box_exact(const LeafRegs& g, const LeafGeo* geo, uint32_t leaf, V3 o, V3 inv,
                                          float tmin, float tmax) {
    const VF4 g3 = ((GlobalF4*)(uintptr_t)(geo + leaf))[3];
    const float x0 = (g.g2[2] - o.x) * inv.x, x1 = (g3[1] - o.x) * inv.x;
    const float y0 = (g.g2[3] - o.y) * inv.y, y1 = (g3[2] - o.y) * inv.y;
    const float z0 = (g3[0] - o.z) * inv.z, z1 = (g3[3] - o.z) * inv.z;
    const float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
    const float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tmax));
    return tn <= tf * kRobust;
}
__device__ __forceinline__ bool leaf_non_opaque(const LeafRegs& r) {
    return (__float_as_uint(r.g2[1]) & kLeafNonOpaque) != 0u;
}
// Any-hit test of a non-opaque leaf hit at barycentric numerators (un, vn) / det by the
// ray (o, d) of a job: whether its surface is present for that ray.
// (Scene: JobRec or BvhView.)
template <class Scene>
__device__ __forceinline__ bool leaf_present(const Scene& J, uint32_t leaf, float un, float vn, float det, V3 o,
                                             V3 d) {
    const MaterialRec& M = J.materials[J.leaf_shade[leaf].material];
    return surface_present(M, J.tex, J.leaf_uv, leaf, un / det, vn / det, opacity_random(J.seed, o, d));
}

// Moller-Trumbore with division-free barycentric acceptance; t = tn / det.
__device__ __forceinline__ bool tri_test(const LeafRegs& g, V3 o, V3 d, float* t_out, float* un_out, float* vn_out,
                                         float* det_out) {
    V3 v0 = v3(g.g0[0], g.g0[1], g.g0[2]);
    V3 e1 = v3(g.g0[3], g.g1[0], g.g1[1]);
    V3 e2 = v3(g.g1[2], g.g1[3], g.g2[0]);
    V3 pv = cross(d, e2);
    float det = dot(e1, pv);
    if (det == 0.0f) return false;
    V3 tv = o - v0;
    float un = dot(tv, pv);
    V3 qv = cross(tv, e1);
    float vn = dot(d, qv);
    if (det > 0.0f) {
        if (un < 0.0f || vn < 0.0f || un + vn > det) return false;
    } else {
        if (un > 0.0f || vn > 0.0f || un + vn < det) return false;
    }
    float tn = dot(e2, qv);
    *t_out = tn / det;
    *un_out = un;
    *vn_out = vn;
    *det_out = det;
    return true;
}
// A lane's traversal stack: the bottom L entries in its LDS column (B ints apart), deeper
// ones in a private array.  A node step pushes at most three entries and pops one; while
// every lane of the wavefront keeps them within the LDS part (`shallow`, one ballot per
// step), a push is one LDS write and one addition, with no check of its own and no
// private-memory access (whose wait would also wait for the node loads).  `top` is the
// lane's next free entry, kept by the caller in a register, apart from the spill array (an
// array indexed at run time is placed in private memory, and a counter beside it would
// follow it there).
typedef __attribute__((address_space(3))) int LdsInt;
template <int L, int B = 256>
struct ShortStack {
    int spill[kStackMax - L];
    LdsInt* bottom;
    __device__ __forceinline__ bool shallow(LdsInt* top) const { return __ballot(top > bottom + (L - 3) * B) == 0ull; }
    __device__ __forceinline__ bool push(LdsInt*& top, int x) {   // any depth
        const int sp = (int)(top - bottom) / B;
        if (sp >= kStackMax) return false;
        if (sp < L) *top = x;
        else spill[sp - L] = x;
        top += B;
        return true;
    }
    __device__ __forceinline__ int pop(LdsInt*& top) {   // any depth
        top -= B;
        const int sp = (int)(top - bottom) / B;
        return sp < L ? *top : spill[sp - L];
    }
};

// Ray fetch for the lanes that ask (the caller decides when a wavefront refills: once
// `refill` lanes are idle, or no lane is busy).  The rays are split into `parts` contiguous
// parts; a wavefront starts on the part of its workgroup's XCD (workgroups go to the XCDs
// round-robin).
//
// Shared parts: each part has a counter on its own 128-B line, one atomic per refill, and a
// wavefront moves on to the following parts when its part runs dry, so no single counter
// sees every refill.
//
// Own runs (no counters, no atomics, nothing that two launches could share): wavefront w of
// a part takes the part's rays 64 w .. 64 w + 63, then those a whole row of wavefronts
// further on, so that neighbouring rays (of like cost, reading like nodes) are spread over the
// wavefronts of the XCD.  Launches without counters (`work` null) deal their rays out that
// way, and so do launches whose wavefronts hold every ray at once; those deal thinly, 8 to
// 64 rays each on about one wavefront per SIMD, because a step of a wavefront with few rays
// waits for fewer cache lookups.  Box room, 320x240, 1 spp, depth 4 (launches of 77k rays
// and fewer): frame 783 -> 663 us.  Queries: 64 rays 55 -> 39 us (of it the scratch's four
// small launches), 2.07 M reflection rays 443 -> 413 us; with one contiguous range per
// wavefront 508 us (ranges of unlike cost); 1.84 M occlusion rays of 2 m, before one ray per
// lane in a plain loop, 458 -> 261 us.
//
// Returns the new ray index for a lane that asked and got one, kNoRay otherwise; nothing is
// left once `left` is 0.
struct WorkCursor {
    uint32_t part;    // part the wavefront draws from
    uint32_t left;    // parts not yet found empty
    uint32_t parts;
    uint32_t chunk;   // rays per part (the last parts may hold fewer)
    bool own;         // own runs of the part
    uint32_t next;    // rays of its runs already taken
    uint32_t run;     // rays per run (64 unless there is only one)
    uint32_t first;   // the first run's offset in the part
    uint32_t row;     // from one run to the next
};
constexpr uint32_t kThinWaves = 1024;   // one wavefront per SIMD
template <int B>
__device__ __forceinline__ WorkCursor work_cursor(const uint32_t* work, uint32_t count, uint32_t parts) {
    const uint32_t chunk = (count + parts - 1u) / parts, part = blockIdx.x % parts;
    const uint32_t waves = gridDim.x / parts * (B / 64);   // a part's (at least one workgroup per part)
    const uint32_t thin = min(64u, max(8u, (count + kThinWaves - 1u) / kThinWaves));
    const bool fits = (uint64_t)thin * waves >= chunk;
    if (!fits && work) return WorkCursor{part, parts, parts, chunk, false, 0u, 0u, 0u, 0u};
    const uint32_t run = fits ? thin : 64u;
    // (a last, incomplete row of workgroups has nothing to do)
    const uint32_t wave = blockIdx.x / parts * (B / 64) +
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t first = wave * run;
    const bool any = wave < waves && first < chunk;
    return WorkCursor{part, any ? 1u : 0u, parts, chunk, true, 0u, run, first, waves * run};
}
__device__ __forceinline__ uint32_t fetch_ray(uint32_t* work, uint32_t count, bool want, WorkCursor& wc) {
    const uint64_t m = __ballot(want);
    if (m == 0ull) return kNoRay;
    const uint32_t lane = __lane_id();
    const uint32_t leader = (uint32_t)__builtin_ctzll(m);
    const uint32_t rank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    if (wc.own) {
        // (one run: next + rank may pass its end; several: runs are 64 rays)
        const uint32_t k = wc.next + rank, turn = k >> 6;
        const bool mine = wc.run == 64u || k < wc.run;
        const uint32_t in_part = wc.first + turn * wc.row + (k & 63u), idx = wc.part * wc.chunk + in_part;
        wc.next += (uint32_t)__popcll(m);
        if ((wc.run != 64u && wc.next >= wc.run) || wc.first + (wc.next >> 6) * wc.row >= wc.chunk) wc.left = 0u;
        return want && mine && in_part < wc.chunk && idx < count ? idx : kNoRay;
    }
    while (wc.left != 0u) {
        const uint32_t lo = min(wc.part * wc.chunk, count);
        const uint32_t hi = min(lo + wc.chunk, count);
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(work + wc.part * kWorkStride, (uint32_t)__popcll(m));
        base = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)leader);
        if (base < hi - lo) {
            const uint32_t idx = base + rank;
            return (want && idx < hi - lo) ? lo + idx : kNoRay;
        }
        wc.part = wc.part + 1u == wc.parts ? 0u : wc.part + 1u;
        --wc.left;
    }
    return kNoRay;
}

// Deferred leaf tests.  A box step does not intersect the leaves it reaches: it appends
// (leaf, owner lane) to its wavefront's queue in LDS, and the queue is flushed -- 64
// tests at a time, one per lane, each lane testing a leaf of any owner with the
// owner's ray fetched by a cross-lane read -- once it holds a test for every busy lane,
// before lanes take new rays, or when no lane has a node left to visit.  So the
// triangle tests run with full wavefronts instead of the few lanes that reach a leaf
// in a given step.  A closest-hit candidate is accepted only where its leaf's own box
// passes the slab test up to the candidate's distance t.  Boxes nest and the slab
// arithmetic rounds monotonically, so every ancestor box of an accepted candidate then
// passes for any running distance >= t: each accepted candidate is reached whatever the
// pruning schedule, and the closest hit -- the minimum of (t, leaf) over accepted
// candidates -- does not depend on when or in which order leaves are tested.  An
// occlusion is an OR over leaves tested against a fixed extent.  A deferred hit only
// prunes later box tests a little later.
constexpr uint32_t kLeafQueue = 64u + 4u * 64u;   // < 64 before a step, which adds <= 4 per lane

// Queue length at which a wavefront with the lanes `busy` visiting nodes tests its queued
// leaves: one leaf per busy lane, at least 8.  A full wavefront waits for 64 tests, so that
// they fill it; a wavefront whose rays are running out (the tail of every launch, and small
// launches throughout) would never gather 64 and its lanes would walk on without the hits
// that end them or shorten them.  Atrium at 1080p, 1 spp: closest hit 2.24 -> 1.95 ms and
// shadow rays 2.15 -> 1.76 ms per frame against waiting for 64; at 16 spp 17.5 -> 17.2 and
// 12.9 -> 12.6 ms.  1.5 or 2 leaves per busy lane: 0.5% slower; half a leaf: 3% slower.
__device__ __forceinline__ uint32_t flush_at(uint64_t busy) { return min(64u, max(8u, (uint32_t)__popcll(busy))); }

// Pointer held by another lane.
template <class T>
__device__ __forceinline__ T* shfl_ptr(T* p, int src) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, src), hi = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src);
    return reinterpret_cast<T*>(((uint64_t)hi << 32) | lo);
}

// Appends the leaf child `link` of the lanes marked in m, with its owner, to the
// wavefront's queue of length qn (uniform).
__device__ __forceinline__ void append_leaf(uint2* queue, uint32_t& qn, bool bit, int link, uint32_t lane) {
    const uint64_t m = __ballot(bit);
    if (bit) {
        const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, qn));
        queue[at] = make_uint2((uint32_t)link, lane);
    }
    qn += (uint32_t)__popcll(m);
}

// One step of every lane that visits a node (cur >= 0): the four child boxes are tested,
// the hit leaves queued, the hit internal child entered nearest (NEAREST) or farthest
// along the ray becomes the next node and the others are pushed in slot order; with none,
// the next node comes from the stack (none left: kParked).
//
// The arithmetic runs for the whole wavefront (idle lanes on whatever their node registers
// hold, their results masked), so that the masks stay in scalar registers and nothing is
// merged at the end of a divergent region; only the loads are under the lanes' mask.
template <bool NEAREST, bool SMALL, int L, int B>
__device__ __forceinline__ void node_step(const TravNode* nodes, int& cur, const TravRay& ray, float tmax,
                                          ShortStack<L, B>& st, LdsInt*& top, uint2* queue, uint32_t& qn, uint32_t lane,
                                          uint32_t* error) {
    const bool busy = cur >= 0;
    NodeRegs n;
    asm volatile("" : "=v"(n.n0), "=v"(n.n1), "=v"(n.n2), "=v"(n.ch));   // any value: masked below
    if (busy) load_node<SMALL>(n, nodes, cur);
    const TravPlanes p = node_planes(n, ray);
    bool in[4], leaf[4];
    float tn[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const bool h = busy & trav_visit(p, k, tmax, &tn[k]);
        in[k] = h & (n.ch[k] > 0);     // an empty slot's link is 0, the root, no node's child
        leaf[k] = h & (n.ch[k] < 0);
    }
    // the entered child: the first of the best; upd[k]: child k was the best so far
    float tb = NEAREST ? (in[0] ? tn[0] : __builtin_inff()) : (in[0] ? tn[0] : -1.0f);
    int next = n.ch[0];
    bool upd[4];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        upd[k] = in[k] & (NEAREST ? tn[k] < tb : tn[k] > tb);
        if (k < 3) tb = upd[k] ? tn[k] : tb;
        next = upd[k] ? n.ch[k] : next;
    }
    const bool none = busy & !(in[0] | in[1] | in[2] | in[3]);
    const bool push[4] = {bool(in[0] & (upd[1] | upd[2] | upd[3])), bool(in[1] & !(upd[1] & !upd[2] & !upd[3])),
                          bool(in[2] & !(upd[2] & !upd[3])), bool(in[3] & !upd[3])};
    if (st.shallow(top)) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (push[k]) {
                *top = n.ch[k];
                top += B;
            }
        }
        if (none) {
            next = kParked;
            if (top > st.bottom) {
                top -= B;
                next = *top;
            }
        }
    } else {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (ok && push[k]) ok = st.push(top, n.ch[k]);
        if (!ok) {
            atomicOr(error, 1u);
            next = kParked;
        } else if (none) {
            next = top > st.bottom ? st.pop(top) : kParked;
        }
    }
    cur = busy ? next : cur;
#pragma unroll
    for (int k = 0; k < 4; ++k) append_leaf(queue, qn, leaf[k], n.ch[k], lane);
}

// Rays of a wave's paths: camera rays (made here, from the path's pixel and sample) or the
// extension queue; hits go to the wave's hit records.
template <bool PRIMARY>
struct PathRays {
    using Scene = JobRec;
    const TraceArgs& a;
    __device__ __forceinline__ uint32_t count() const { return PRIMARY ? a.jobs.num_paths : *a.count_in; }
    __device__ __forceinline__ const JobRec* scene() const { return a.jobs.rec; }
    template <bool ONE>
    __device__ __forceinline__ const JobRec* start(uint32_t i, V3& o, V3& d, float& tmax) const {
        const uint32_t path = PRIMARY || ONE || a.jobs.num_jobs == 1u ? i : a.q.path[i];
        const JobRec* rec = nullptr;
        with_job<ONE>(a.jobs, path, [&](const JobRec& J, uint32_t local) {
            rec = &J;
            tmax = J.ray_length;
            if constexpr (PRIMARY) {
                const PathKey k = path_key(J, local);
                float jx = 0.5f, jy = 0.5f;
                if (J.flags & 1u) {
                    Pcg jr = pcg_keyed(J.seed, k.pixel, k.sample, kJitterBounce);
                    jx = pcg_float(jr);
                    jy = pcg_float(jr);
                }
                camera_ray(J.cam, k.pixel % J.cam.width, k.pixel / J.cam.width, jx, jy, &o, &d);
            }
        });
        if constexpr (!PRIMARY) {
            o = v3(a.q.ox[i], a.q.oy[i], a.q.oz[i]);
            d = v3(a.q.dx[i], a.q.dy[i], a.q.dz[i]);
        }
        return rec;
    }
    __device__ __forceinline__ void finish(uint32_t i, HitRec h) const { a.hits.rec[i] = h; }
};
// Rays of a query (the caller's arrays); results go straight to the caller's arrays: t (+inf
// on a miss), the triangle's index in the scene's order, barycentrics; or whether anything
// was hit.
struct QueryRays {
    using Scene = BvhView;
    const QueryArgs& a;
    __device__ __forceinline__ uint32_t count() const { return a.count; }
    __device__ __forceinline__ const BvhView* scene() const { return &a.bvh; }
    template <bool ONE>
    __device__ __forceinline__ const BvhView* start(uint32_t i, V3& o, V3& d, float& tmax) const {
        o = v3(a.q.ox[i], a.q.oy[i], a.q.oz[i]);
        d = v3(a.q.dx[i], a.q.dy[i], a.q.dz[i]);
        tmax = a.tmax;
        return &a.bvh;
    }
    __device__ __forceinline__ void finish(uint32_t i, HitRec h) const {
        const bool hit = h.leaf != kLeafMiss;
        if (a.t) a.t[i] = hit ? h.t : __builtin_inff();
        a.triangle[i] = hit && a.order ? a.order[h.leaf] : h.leaf;
        if (a.u) a.u[i] = h.u;
        if (a.v) a.v[i] = h.v;
    }
    __device__ __forceinline__ void finish_any(uint32_t i, bool occ) const { a.triangle[i] = occ ? 1u : 0u; }
};

// AH: the call's scenes hold non-opaque (alpha-tested or translucent) triangles, whose
// hits pass the any-hit test; without them the test and its registers are compiled out.
// ONE: every ray of the launch belongs to one scene whose nodes lie within 4 GB, so the
// scene pointers are uniform (scalar registers) instead of per lane.
// S: where rays come from and hits go (PathRays, QueryRays): the scene of ray 0, a ray's
// origin, direction, extent and scene, and its finished hit.
template <bool AH, int L, int B, bool ONE, class S>
__device__ __forceinline__ void trace_closest_body(const S& src, const TraceLoop& a) {
    __shared__ int lds[L][B];
    __shared__ uint2 s_queue[B / 64][kLeafQueue];
    __shared__ unsigned long long s_key[B / 64][64];
    __shared__ float2 s_uv[B / 64][64];
    const uint32_t count = src.count();
    const float tmin = kTMin;
    // Each lane keeps its ray's scene (BVH nodes, leaf records, triangle count): a wave
    // may hold rays of several jobs.  A job without triangles points at a one-node tree
    // whose slots are all empty.
    // Each iteration: (1) lanes with a node to visit test its four child boxes, push the
    // hit internal children but the nearest, queue the hit leaves and move to the
    // nearest (a lane with nothing left is parked until its queued leaves are tested);
    // (2) the leaf queue is flushed at flush_at, before a refill, or when no lane is busy,
    // and parked lanes with no queued leaves write their hit; (3) idle lanes take new
    // rays (starting at the root) once enough of them are idle.  The best hit of a lane's
    // ray sits in LDS: key (t bits, leaf), the smaller the better, and the barycentrics,
    // written by the lane that tested the winning leaf.
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    uint2* queue = s_queue[w];
    unsigned long long* key = s_key[w];
    float2* uv = s_uv[w];
    uint32_t qn = 0;
    uint32_t ray = kNoRay;
    WorkCursor wc = work_cursor<B>(a.work, count, a.parts);
    V3 o = v3(0.f, 0.f, 0.f), d = v3(0.f, 0.f, 1.f);
    TravRay rb = trav_ray(o, d);
    float tbest = 0.0f;
    const typename S::Scene* scene = src.scene();   // the lane's scene (materials for any-hit tests)
    const TravNode* nodes = scene->nodes;
    const LeafGeo* geo = scene->leaf_geo;
    ShortStack<L, B> st;
    st.bottom = (LdsInt*)&lds[0][threadIdx.x];
    LdsInt* top = st.bottom;
    int cur = kIdle;
    uint32_t dry = 0;   // steps since a ray of the wavefront finished
    for (;;) {
        node_step<true, ONE, L, B>(nodes, cur, rb, tbest, st, top, queue, qn, lane, a.error);
        // a ray enters each node at most once: more steps than nodes with no ray finished
        // means corrupt links, and the rays are ended instead of looping
        if (++dry > a.step_bound) {
            if (lane == 0) atomicOr(a.error, 8u);
            if (cur >= 0) cur = kParked;
        }
        const uint64_t busy = __ballot(cur >= 0);
        const bool refill_now =
            wc.left != 0u && (busy == 0ull || 64u - (uint32_t)__popcll(busy) >= a.refill);
        if (qn != 0u && (qn >= flush_at(busy) || refill_now || busy == 0ull)) {
            __builtin_amdgcn_wave_barrier();
            for (uint32_t b = 0; b < qn; b += 64u) {
                const uint32_t e = b + lane;
                const bool valid = e < qn;
                const uint2 q = valid ? queue[e] : make_uint2(~0u, lane);
                const uint32_t leaf = ~q.x;
                const int owner = (int)q.y;
                const V3 oo = v3(__shfl(o.x, owner), __shfl(o.y, owner), __shfl(o.z, owner));
                const V3 dd = v3(__shfl(d.x, owner), __shfl(d.y, owner), __shfl(d.z, owner));
                const V3 oi = v3(__shfl(rb.inv[0], owner), __shfl(rb.inv[1], owner), __shfl(rb.inv[2], owner));
                const float tb = __shfl(tbest, owner);
                const LeafGeo* og = ONE ? geo : shfl_ptr(geo, owner);
                // a hit counts only where the leaf's own box passes the slab test up to the
                // hit distance (the acceptance rule that makes the closest hit independent
                // of the order leaves are found in), and, for a non-opaque leaf, where its
                // surface is present for the ray (a function of the ray and the leaf alone)
                float t = 0.0f, un = 0.0f, vn = 0.0f, det = 1.0f;
                LeafRegs lr{};
                if (valid) lr = load_leaf(og, leaf);
                bool cand = valid && tri_test(lr, oo, dd, &t, &un, &vn, &det) && t >= tmin && t <= tb &&
                            box_exact(lr, og, leaf, oo, oi, tmin, t);
                if constexpr (AH) {
                    const bool nop = cand && leaf_non_opaque(lr);
                    if (__ballot(nop) != 0ull) {
                        const typename S::Scene* os = ONE ? scene : shfl_ptr(scene, owner);
                        if (nop) cand = leaf_present(*os, leaf, un, vn, det, oo, dd);
                    }
                }
                const unsigned long long mine = ((unsigned long long)__float_as_uint(t) << 32) | leaf;
                if (cand) atomicMin(&key[owner], mine);
                __builtin_amdgcn_wave_barrier();
                if (cand && key[owner] == mine) uv[owner] = make_float2(un / det, vn / det);
            }
            __builtin_amdgcn_wave_barrier();
            qn = 0;
            tbest = __uint_as_float((uint32_t)(key[lane] >> 32));
        }
        if (qn == 0u && __ballot(cur == kParked) != 0ull) {   // rays whose leaves are all tested: write the hits
            dry = 0;
            if (cur == kParked) {
                const float2 buv = uv[lane];
                src.finish(ray, HitRec{tbest, (uint32_t)key[lane], buv.x, buv.y});
                cur = kIdle;
            }
        }
        uint32_t got = kNoRay;
        if (refill_now) got = fetch_ray(a.work, count, cur == kIdle, wc);
        const bool fresh = got != kNoRay;
        if (fresh) {
            float tmax = 0.0f;
            const typename S::Scene* sc = src.template start<ONE>(got, o, d, tmax);
            if constexpr (!ONE) {
                scene = sc;
                nodes = sc->nodes;
                geo = sc->leaf_geo;
            }
            ray = got;
            rb = trav_ray(o, d);
            tbest = tmax;
            key[lane] = ((unsigned long long)__float_as_uint(tmax) << 32) | kLeafMiss;
            uv[lane] = make_float2(0.0f, 0.0f);
            top = st.bottom;
            cur = 0;
        }
        if (wc.left == 0u && __ballot(cur != kIdle) == 0ull) break;
    }
}

template <bool PRIMARY, bool AH, int L, int B>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(AH ? 4 : 6))) void k_trace_closest(TraceArgs a) {
    trace_closest_body<AH, L, B, false>(PathRays<PRIMARY>{a}, a.loop);
}
// One job, opaque scene, 256-thread blocks and a 12-deep LDS stack (the defaults): the
// scene pointers sit in scalar registers, which frees six vector registers per lane.
template <bool PRIMARY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_trace_closest_one(TraceArgs a) {
    trace_closest_body<false, 12, 256, true>(PathRays<PRIMARY>{a}, a.loop);
}
template <bool AH, bool ONE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(AH ? 5 : 6))) void k_query_closest(QueryArgs a) {
    trace_closest_body<AH, 12, 256, ONE>(QueryRays{a}, a.loop);
}

// Adds shadow ray i's contribution unless it is occluded; returns whether it is a sky ray.
__device__ __forceinline__ bool apply_shadow(const ShadowArgs& a, uint32_t i, bool occ) {
    const float4 cp = a.q.cp[i];
    const uint32_t pk = shadow_pk(cp), path = pk >> 3, kind = pk & 7u;
    V3 c = v3(cp.x, cp.y, cp.z);
    if (occ) {
        if (kind == kKindSky) return true;
        if (!a.any_keep) return false;   // no light of the launch shines through its shadow
        const uint32_t job = a.jobs.num_jobs == 1u ? 0u : job_of(a.jobs.path_base, a.jobs.num_jobs, path);
        const float keep = a.jobs.rec[job].keep[kind];
        if (!(keep > 0.0f)) return false;
        c = c * keep;
    }
    const uint32_t slot = kind == kKindSky ? kSlotSky : kSlotLights + kind;
    Rgb* acc = a.ps.acc + (size_t)slot * a.ps.cap + path;
    const Rgb s = *acc;
    *acc = Rgb{s.x + c.x, s.y + c.y, s.z + c.z};
    return kind == kKindSky;
}

// A segment's shadow rays; a finished ray adds its contribution to its path.
struct ShadowRays {
    using Scene = JobRec;
    const ShadowArgs& a;
    uint32_t& sky_rays;   // ray statistics: sky shadow rays this lane finished
    __device__ __forceinline__ uint32_t count() const { return *a.count_in; }
    __device__ __forceinline__ const JobRec* scene() const { return a.jobs.rec; }
    // A sky ray's direction is in the queue; a light's ray is rebuilt from the light as the
    // shading built it (without point lights, every light is directional and every extent
    // unbounded).
    template <bool AH, bool ONE>
    __device__ __forceinline__ const JobRec* start(uint32_t i, V3& o, V3& d, float& tmax) const {
        const uint32_t pk = shadow_pk(a.q.cp[i]), kind = pk & 7u;
        o = v3(a.q.ox[i], a.q.oy[i], a.q.oz[i]);
        tmax = kShadowTMax;
        const JobRec* rec = nullptr;
        with_job<ONE>(a.jobs, pk >> 3, [&](const JobRec& J, uint32_t) {
            rec = &J;
            if (kind == kKindSky) {
                d = v3(a.q.dx[i], a.q.dy[i], a.q.dz[i]);
            } else if constexpr (AH) {
                light_shadow_ray(J.lights[kind], o, &d, &tmax);
            } else {
                const LightRec& Lk = J.lights[kind];
                d = v3(Lk.direction[0], Lk.direction[1], Lk.direction[2]);
            }
        });
        return rec;
    }
    __device__ __forceinline__ void finish_any(uint32_t i, bool occ) const { sky_rays += apply_shadow(a, i, occ) ? 1u : 0u; }
};
// Rays of an occlusion query.
struct AnyQueryRays : QueryRays {
    template <bool AH, bool ONE>
    __device__ __forceinline__ const BvhView* start(uint32_t i, V3& o, V3& d, float& tmax) const {
        return QueryRays::start<ONE>(i, o, d, tmax);
    }
};

// AH (the general variant): any-hit tests of non-opaque leaves and rays of finite extent
// (towards point lights, occlusion queries); launched when a scene of the call has either.
template <bool AH, int L, int B, bool ONE, class S>
__device__ __forceinline__ void trace_any_body(const S& src, const TraceLoop& a) {
    __shared__ int lds[L][B];
    __shared__ uint2 s_queue[B / 64][kLeafQueue];
    __shared__ uint32_t s_occ[B / 64][64];
    const uint32_t count = src.count();
    const float tmin = kTMin;
    // a ray's extent: unbounded towards the sky and directional lights, the distance to a
    // point light or a query's (the general variant only)
    float tmax = kShadowTMax;
    // Same iteration as the closest-hit kernel: box steps queue their leaves, the queue
    // is flushed at flush_at, before a refill or when no lane is busy, and parked lanes
    // finish once their leaves are tested.  The hit internal child whose box the ray enters
    // farthest away is entered (occluders are found sooner there than near the ray's own
    // surface: C1 shadow rays visit 8.9 nodes instead of 11.3 in slot order) and the others
    // pushed in slot order (the answer is order-independent).  A flush that finds a ray
    // occluded ends it at once, busy or parked.
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    uint2* queue = s_queue[w];
    uint32_t* occf = s_occ[w];
    occf[lane] = 0u;
    uint32_t qn = 0;
    uint32_t ray = kNoRay;
    WorkCursor wc = work_cursor<B>(a.work, count, a.parts);
    V3 o = v3(0.f, 0.f, 0.f), d = v3(0.f, 0.f, 1.f);
    TravRay rb = trav_ray(o, d);
    const typename S::Scene* scene = src.scene();   // the lane's ray's scene (see trace_closest_body)
    const TravNode* nodes = scene->nodes;
    const LeafGeo* geo = scene->leaf_geo;
    ShortStack<L, B> st;
    st.bottom = (LdsInt*)&lds[0][threadIdx.x];
    LdsInt* top = st.bottom;
    int cur = kIdle;
    uint32_t dry = 0;   // steps since a ray of the wavefront finished
    for (;;) {
        node_step<false, ONE, L, B>(nodes, cur, rb, tmax, st, top, queue, qn, lane, a.error);
        if (++dry > a.step_bound) {   // corrupt links (see k_trace_closest)
            if (lane == 0) atomicOr(a.error, 8u);
            if (cur >= 0) cur = kParked;
        }
        const uint64_t busy = __ballot(cur >= 0);
        const bool refill_now =
            wc.left != 0u && (busy == 0ull || 64u - (uint32_t)__popcll(busy) >= a.refill);
        bool occ = false;
        if (qn != 0u && (qn >= flush_at(busy) || refill_now || busy == 0ull)) {
            __builtin_amdgcn_wave_barrier();
            for (uint32_t b = 0; b < qn; b += 64u) {
                const uint32_t e = b + lane;
                const bool valid = e < qn;
                const uint2 q = valid ? queue[e] : make_uint2(~0u, lane);
                const uint32_t leaf = ~q.x;
                const int owner = (int)q.y;
                const V3 oo = v3(__shfl(o.x, owner), __shfl(o.y, owner), __shfl(o.z, owner));
                const V3 dd = v3(__shfl(d.x, owner), __shfl(d.y, owner), __shfl(d.z, owner));
                const V3 oi = v3(__shfl(rb.inv[0], owner), __shfl(rb.inv[1], owner), __shfl(rb.inv[2], owner));
                const LeafGeo* og = ONE ? geo : shfl_ptr(geo, owner);
                float t = 0.0f, un = 0.0f, vn = 0.0f, det = 1.0f;
                LeafRegs lr{};
                if (valid) lr = load_leaf(og, leaf);
                const float tm = AH ? __shfl(tmax, owner) : kShadowTMax;
                bool cand = valid && tri_test(lr, oo, dd, &t, &un, &vn, &det) && t >= tmin && t <= tm &&
                            box_exact(lr, og, leaf, oo, oi, tmin, tm);
                if constexpr (AH) {
                    const bool nop = cand && leaf_non_opaque(lr);
                    if (__ballot(nop) != 0ull) {
                        const typename S::Scene* os = ONE ? scene : shfl_ptr(scene, owner);
                        if (nop) cand = leaf_present(*os, leaf, un, vn, det, oo, dd);
                    }
                }
                if (cand) occf[owner] = 1u;
            }
            __builtin_amdgcn_wave_barrier();
            qn = 0;
            occ = occf[lane] != 0u;
            if (occ) occf[lane] = 0u;
        }
        const bool done = cur != kIdle && (occ || (cur == kParked && qn == 0u));
        if (__ballot(done) != 0ull) {
            dry = 0;
            if (done) {
                src.finish_any(ray, occ);
                cur = kIdle;
            }
        }
        uint32_t got = kNoRay;
        if (refill_now) got = fetch_ray(a.work, count, cur == kIdle, wc);
        const bool fresh = got != kNoRay;
        if (fresh) {
            float extent;
            const typename S::Scene* sc = src.template start<AH, ONE>(got, o, d, extent);
            if constexpr (AH) tmax = extent;
            if constexpr (!ONE) {
                scene = sc;
                nodes = sc->nodes;
                geo = sc->leaf_geo;
            }
            ray = got;
            rb = trav_ray(o, d);
            top = st.bottom;
            cur = 0;
        }
        if (wc.left == 0u && __ballot(cur != kIdle) == 0ull) break;
    }
}

template <bool AH, int L, int B, bool ONE>
__device__ __forceinline__ void trace_shadow(const ShadowArgs& a) {
    uint32_t sky_rays = 0;
    trace_any_body<AH, L, B, ONE>(ShadowRays{a, sky_rays}, a.loop);
    // the shade launch counted every shadow ray as a light shadow ray: move the sky
    // rays over, one atomic pair per workgroup
    for (int off = 32; off >= 1; off >>= 1) sky_rays += __shfl_xor(sky_rays, off);
    __shared__ uint32_t s_sky[B / 64];
    if (__lane_id() == 0) s_sky[threadIdx.x >> 6] = sky_rays;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int k = 0; k < B / 64; ++k) tot += s_sky[k];
        if (tot) {
            atomicAdd(reinterpret_cast<unsigned long long*>(a.ray_counters + 2), (unsigned long long)(0ull - tot));
            atomicAdd(reinterpret_cast<unsigned long long*>(a.ray_counters + 3), (unsigned long long)tot);
        }
    }
}

template <bool AH, int L, int B>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(AH ? 5 : 6))) void k_trace_shadow(ShadowArgs a) {
    trace_shadow<AH, L, B, false>(a);
}
// One job, opaque scene, the default stack and block (as k_trace_closest_one).
__global__ __launch_bounds__(256) void k_trace_shadow_one(ShadowArgs a) { trace_shadow<false, 12, 256, true>(a); }
// Occlusion queries: their extent is the caller's, so the general variant.
template <bool ONE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ONE ? 6 : 5))) void k_query_any(QueryArgs a) {
    trace_any_body<true, 12, 256, ONE>(AnyQueryRays{{a}}, a.loop);
}

// Workgroups that stay resident on the whole chip for a kernel (persistent grid).
template <class K>
uint32_t resident_groups(K kernel, int block) {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
    }
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess || per_cu <= 0)
        per_cu = 1024 / block;
    return (uint32_t)(cus * per_cu);
}

// Workgroups of a launch of up to n rays: at least those that deal few rays out thinly
// (work_cursor), at most what stays resident, in whole rows of one workgroup per part.
template <int B, class K>
uint32_t launch_groups(K kernel, uint32_t& resident, uint32_t n, uint32_t parts) {
    if (resident == 0) resident = resident_groups(kernel, B);
    constexpr uint32_t per = B / 64;
    const uint32_t thin = std::min((n + 8u * per - 1u) / (8u * per), kThinWaves / per);
    const uint32_t rows = (std::max((n + B - 1u) / B, thin) + parts - 1u) / parts;
    return std::max(std::min(rows, resident / parts), 1u) * parts;
}

template <bool P, bool AH, int L, int B>
void closest_lb(const TraceArgs& a, uint32_t capacity, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<B>(k_trace_closest<P, AH, L, B>, resident, capacity, a.loop.parts);
    hipLaunchKernelGGL((k_trace_closest<P, AH, L, B>), dim3(groups), dim3(B), 0, s, a);
}

template <bool P>
void closest_one(const TraceArgs& a, uint32_t capacity, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<256>(k_trace_closest_one<P>, resident, capacity, a.loop.parts);
    hipLaunchKernelGGL((k_trace_closest_one<P>), dim3(groups), dim3(256), 0, s, a);
}

void shadow_one(const ShadowArgs& a, uint32_t capacity, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<256>(k_trace_shadow_one, resident, capacity, a.loop.parts);
    hipLaunchKernelGGL(k_trace_shadow_one, dim3(groups), dim3(256), 0, s, a);
}

template <bool AH, int L, int B>
void shadow_lb(const ShadowArgs& a, uint32_t capacity, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<B>(k_trace_shadow<AH, L, B>, resident, capacity, a.loop.parts);
    hipLaunchKernelGGL((k_trace_shadow<AH, L, B>), dim3(groups), dim3(B), 0, s, a);
}

// Block shapes: 128, 256 (default) or 512 threads; LDS stack depths 8, 12 (default), 16, 24, 32.
template <bool P, bool AH, int B>
void closest_b(const TraceArgs& a, uint32_t capacity, uint32_t lds, hipStream_t s) {
    if (lds <= 8) closest_lb<P, AH, 8, B>(a, capacity, s);
    else if (lds <= 12) closest_lb<P, AH, 12, B>(a, capacity, s);
    else if (lds <= 16) closest_lb<P, AH, 16, B>(a, capacity, s);
    else if (lds <= 24) closest_lb<P, AH, 24, B>(a, capacity, s);
    else closest_lb<P, AH, 32, B>(a, capacity, s);
}

template <bool P, bool AH>
void dispatch_closest(const TraceArgs& a, uint32_t capacity, uint32_t lds, uint32_t block, hipStream_t s) {
    if (block == 128) closest_b<P, AH, 128>(a, capacity, lds, s);
    else if (block == 512) closest_b<P, AH, 512>(a, capacity, lds, s);
    else closest_b<P, AH, 256>(a, capacity, lds, s);
}

template <bool AH, int B>
void shadow_b(const ShadowArgs& a, uint32_t capacity, uint32_t lds, hipStream_t s) {
    if (lds <= 8) shadow_lb<AH, 8, B>(a, capacity, s);
    else if (lds <= 12) shadow_lb<AH, 12, B>(a, capacity, s);
    else if (lds <= 16) shadow_lb<AH, 16, B>(a, capacity, s);
    else if (lds <= 24) shadow_lb<AH, 24, B>(a, capacity, s);
    else shadow_lb<AH, 32, B>(a, capacity, s);
}

template <bool AH>
void dispatch_shadow(const ShadowArgs& a, uint32_t capacity, uint32_t lds, uint32_t block, hipStream_t s) {
    if (block == 128) shadow_b<AH, 128>(a, capacity, lds, s);
    else if (block == 512) shadow_b<AH, 512>(a, capacity, lds, s);
    else shadow_b<AH, 256>(a, capacity, lds, s);
}

}  // namespace

void launch_trace_closest(const TraceArgs& a, uint32_t capacity, bool primary, uint32_t lds_stack, uint32_t block,
                          hipStream_t s) {
    if (capacity == 0) return;
    if (a.loop.one && !a.loop.any_hit && block == 256 && lds_stack > 8 && lds_stack <= 12) {
        if (primary) closest_one<true>(a, capacity, s);
        else closest_one<false>(a, capacity, s);
        return;
    }
    if (primary) {
        if (a.loop.any_hit) dispatch_closest<true, true>(a, capacity, lds_stack, block, s);
        else dispatch_closest<true, false>(a, capacity, lds_stack, block, s);
    } else {
        if (a.loop.any_hit) dispatch_closest<false, true>(a, capacity, lds_stack, block, s);
        else dispatch_closest<false, false>(a, capacity, lds_stack, block, s);
    }
}

namespace {

template <bool AH, bool ONE>
void query_closest(const QueryArgs& a, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<256>(k_query_closest<AH, ONE>, resident, a.count, a.loop.parts);
    hipLaunchKernelGGL((k_query_closest<AH, ONE>), dim3(groups), dim3(256), 0, s, a);
}
template <bool ONE>
void query_any(const QueryArgs& a, hipStream_t s) {
    static uint32_t resident = 0;
    const uint32_t groups = launch_groups<256>(k_query_any<ONE>, resident, a.count, a.loop.parts);
    hipLaunchKernelGGL((k_query_any<ONE>), dim3(groups), dim3(256), 0, s, a);
}

}  // namespace

void launch_query_closest(const QueryArgs& a, hipStream_t s) {
    if (a.count == 0) return;
    if (a.loop.any_hit) a.loop.one ? query_closest<true, true>(a, s) : query_closest<true, false>(a, s);
    else a.loop.one ? query_closest<false, true>(a, s) : query_closest<false, false>(a, s);
}
void launch_query_any(const QueryArgs& a, hipStream_t s) {
    if (a.count == 0) return;
    a.loop.one ? query_any<true>(a, s) : query_any<false>(a, s);
}

void launch_trace_shadow(const ShadowArgs& a, uint32_t capacity, uint32_t lds, uint32_t block, hipStream_t s) {
    if (capacity == 0) return;
    if (a.loop.one && !a.loop.any_hit && block == 256 && lds > 8 && lds <= 12) {
        shadow_one(a, capacity, s);
        return;
    }
    if (a.loop.any_hit) dispatch_shadow<true>(a, capacity, lds, block, s);
    else dispatch_shadow<false>(a, capacity, lds, block, s);
}

}  // namespace bipt
