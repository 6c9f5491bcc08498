// pt_kernels.hpp -- kernel argument blocks and launchers of the path-tracing pass.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pt_device.hpp"
#include "pt_layout.hpp"

namespace bipt {

PT_HD uint32_t expand10(uint32_t v) {
    v &= 1023u;
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}
PT_HD uint32_t morton3(uint32_t x, uint32_t y, uint32_t z) {
    return (expand10(x) << 2) | (expand10(y) << 1) | expand10(z);
}

struct BuildArgs {
    const float* positions;
    const float* normals;
    const uint32_t* indices;
    const InstanceRec* instances;
    uint32_t num_instances;
    uint32_t num_tris;
    float* tri_v;
    float* tri_n;
    uint32_t* tri_mat;
    uint32_t* cbounds_ord;   // bounds_words() words: order-preserving bounds (min xyz, max xyz)
    float* cbounds_out;      // 6 floats (may be null)
    uint32_t* keys[2];
    uint32_t* vals[2];
    uint32_t* sort_counters;   // sort_words(num_tris) words
    BvhNode* nodes;
    TravNode* nodes4;
    int32_t* parent;
    uint32_t* refit_cnt;
    LeafGeo* leaf_geo;
    LeafShade* leaf_shade;
    const MaterialRec* materials;   // blend modes: non-opaque leaves are flagged
    // per-vertex texture coordinates (2 floats) and tangents (4), and the per-leaf copies
    // made from them (all null unless the scene's materials need them)
    const float* uvs;
    const float* tangents;
    LeafUv* leaf_uv;
    LeafTan* leaf_tan;
    uint32_t* error;
    // treelet restructuring after the refit (0 rounds: the Morton/Karras tree as built)
    uint32_t treelet_rounds;
    float* tl_cost;
    int32_t* tl_height;
    int32_t* tl_snap;    // per internal node: height at the start of a round
    uint32_t* tl_starts; // 1 + treelet_start_cap(num_tris) entries
};
void launch_build_lbvh(const BuildArgs& a, hipStream_t s);
uint32_t bounds_words();
uint32_t sort_words(uint32_t n);
uint32_t treelet_start_cap(uint32_t n);

// Jobs of a wave: records, path bases (num_jobs + 1 entries, the last = paths in the
// wave) and pixel bases (num_jobs + 1 entries) for the resolve pass.
struct WaveJobs {
    const JobRec* rec;
    const uint32_t* path_base;
    const uint32_t* pix_base;
    uint32_t num_jobs;
    uint32_t num_paths;
};

// Job of a path (or pixel slot): the last j with base[j] <= x.
PT_HD uint32_t job_of(const uint32_t* base, uint32_t n, uint32_t x) {
    uint32_t lo = 0, hi = n;   // base[lo] <= x < base[hi]
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (base[mid] <= x) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Calls f(job record, path within the job) for each lane's path.  Queues hold paths in
// increasing order, so the lanes of a wavefront nearly always have paths of one job: its
// record is then read at a uniform address (scalar loads), the job found by one scalar
// search.  A wavefront that straddles jobs looks up a job per lane.  ONE: a single job.
// 24-scene batch: 34.7 -> 32.6 ms; radiance-cache frame (image and training jobs): 4.66 ->
// 4.60 ms.
template <bool ONE, class F>
__device__ __forceinline__ void with_job(const WaveJobs& jobs, uint32_t path, F f) {
    if (ONE || jobs.num_jobs == 1u) {
        f(jobs.rec[0], path);
        return;
    }
    const uint32_t p0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)path);
    const uint32_t j0 = job_of(jobs.path_base, jobs.num_jobs, p0);
    const uint32_t lo = jobs.path_base[j0], hi = jobs.path_base[j0 + 1u];
    if (__ballot(path < lo || path >= hi) == 0ull) {
        f(jobs.rec[j0], path - lo);
    } else {
        const uint32_t j = job_of(jobs.path_base, jobs.num_jobs, path);
        f(jobs.rec[j], path - jobs.path_base[j]);
    }
}

// As with_job with one copy of f: the wavefront takes its jobs one after the other, each at
// a uniform address (for code so large that with_job's three copies crowd the instruction
// cache).
template <class F>
__device__ __forceinline__ void each_job(const WaveJobs& jobs, uint32_t path, F f) {
    uint32_t j = jobs.num_jobs == 1u ? 0u : job_of(jobs.path_base, jobs.num_jobs, path);
    for (bool done = false; !done;) {
        const uint32_t j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)j);
        if (j == j0) {
            f(jobs.rec[j0], path - (jobs.num_jobs == 1u ? 0u : jobs.path_base[j0]));
            done = true;
        }
    }
}

// Slot, pixel and sample of a job's local path: images walk their pixels in 8x8 tile
// order, sample after sample; the cache's training paths take one pixel per slot drawn
// uniformly from the image (PCG32 keyed by the job seed and slot) and use the slot as
// their sample index, so no two training paths share a random stream.
constexpr uint32_t kTrainPixelBounce = 254u;
struct PathKey {
    uint32_t q, pixel, sample;
};
PT_HD PathKey path_key(const JobRec& J, uint32_t local) {
    const uint32_t q = local % J.npix, sl = local / J.npix;
    if (J.flags & kJobTrain) {
        Pcg r = pcg_keyed(J.seed, q, 0u, kTrainPixelBounce);
        const uint64_t npix = (uint64_t)J.cam.width * J.cam.height;
        return PathKey{q, (uint32_t)(((uint64_t)pcg_next(r) * npix) >> 32), q};
    }
    return PathKey{q, pixel_of(q, J.cam.width, J.cam.height), J.sample0 + sl};
}

// The traversal loop of a launch: how its persistent lanes share the rays.
struct TraceLoop {
    uint32_t* work;             // part counters of the persistent lanes (zero at launch); null: every
                                // wavefront has its own range of rays
    uint32_t parts;             // queue parts (1..kWorkPartsMax)
    uint32_t refill;            // idle lanes before a refill (1..64)
    uint32_t any_hit;           // nonzero: some scene of the call has non-opaque triangles (shadow
                                // launches: or point lights)
    uint32_t one;               // nonzero: one scene of at most kSmallTreeTris triangles
    uint32_t step_bound;        // steps without a finished ray that only corrupt links can reach (trace_step_bound)
    uint32_t* error;
};
struct TraceArgs {
    WaveJobs jobs;
    RayQueue q;                 // input queue (unused for primary rays)
    const uint32_t* count_in;   // device count (null: primary, count = jobs.num_paths)
    HitBuf hits;
    TraceLoop loop;
};
// A ray enters each node of its tree at most once and then waits for its leaves' tests:
// tris is the most triangles of a scene of the launch.
PT_HD uint32_t trace_step_bound(uint32_t tris) { return tris + 4u; }
// block: threads per workgroup of the persistent grid (128, 256 or 512; else 256).
void launch_trace_closest(const TraceArgs& a, uint32_t capacity, bool primary, uint32_t lds_stack, uint32_t block,
                          hipStream_t s);

// Ray queries: `count` rays of one extent, one scene.
struct QueryArgs {
    BvhView bvh;
    RayQueue q;                 // path unused
    uint32_t count;
    float tmax;
    const uint32_t* order;      // leaf -> triangle (null: the leaf itself)
    float* t;                   // nullable
    uint32_t* triangle;         // or, for occlusion, 1 / 0
    float *u, *v;               // nullable
    TraceLoop loop;
};
void launch_query_closest(const QueryArgs& a, hipStream_t s);
void launch_query_any(const QueryArgs& a, hipStream_t s);

struct ShadowArgs {
    WaveJobs jobs;
    ShadowQueue q;
    const uint32_t* count_in;
    PathState ps;
    uint64_t* ray_counters;     // sky shadow rays move from [2] (all shadow rays) to [3]
    uint32_t any_keep;          // nonzero: some light of the launch keeps a part when occluded (JobRec::keep)
    TraceLoop loop;
};
void launch_trace_shadow(const ShadowArgs& a, uint32_t capacity, uint32_t lds_stack, uint32_t block, hipStream_t s);

// Shading of one segment writes its outputs straight into the next queues, in entry
// order: each 256-entry tile publishes its totals and finds its offset by decoupled
// look-back over the tiles before it.
struct ShadeArgs {
    WaveJobs jobs;
    RayQueue qin;
    const uint32_t* count_in;   // null at bounce 0
    HitBuf hits;
    PathState ps;
    RayQueue qout;              // extension rays of the next segment
    ShadowQueue sq;             // shadow rays of this segment (kinds: lights, then the sky)
    uint32_t* count_ext;        // written by the last tile (zeroed by launch_shade_reset)
    uint32_t* count_shadow;
    uint64_t* ray_counters;     // [camera, extension, light shadow, sky shadow]
    uint64_t* tile_state;       // per tile: look-back word (zero at launch)
    uint32_t* error;            // 32: a look-back wait ran out
    uint32_t* trace_work_reset;   // zeroed here for the next closest-hit launch
    uint32_t* shadow_work_reset;  // zeroed here for this segment's shadow launch
    uint32_t bounce;
    NrcRecord* nrc_query;         // non-null: the cache kernel runs after this segment's
                                  // shading; entry i's query (or kNoPath) goes to [i]
};
// Clears the output counts and the look-back words of the tiles the next shade launch
// covers (count_in entries, or num_entries if count_in is null).
void launch_shade_reset(uint64_t* tile_state, const uint32_t* count_in, uint32_t num_entries, uint32_t* count_ext,
                        uint32_t* count_shadow, uint32_t capacity, hipStream_t s);
// max_lights: the most lights of any job in the launch (at most kMaxDirLights).
void launch_shade(const ShadeArgs& a, uint32_t capacity, uint32_t max_lights, hipStream_t s);

// Rect lights of a segment's vertices (waves where some job has them), after its shading.
struct RectArgs {
    WaveJobs jobs;
    RayQueue qin;
    const uint32_t* count_in;   // null at bounce 0
    HitBuf hits;
    PathState ps;
    uint32_t bounce;
};
void launch_shade_rect(const RectArgs& a, uint32_t capacity, hipStream_t s);

struct ResolveArgs {
    WaveJobs jobs;
    PathState ps;
    uint32_t num_pix;     // resolve slots of the wave (sum of the jobs' pixels)
};
void launch_resolve(const ResolveArgs& a, hipStream_t s);
// Running mean of every job of the wave -> its RGBA32F output.
void launch_output(const WaveJobs& jobs, uint32_t num_pix, hipStream_t s);
// Primary-hit GBuffer of the job record `job` (device) from the segment-0 hit records of its
// paths [path0, path0 + npix): its first sample in the wave, which must be the call's first.
void launch_gbuffer(const JobRec* job, const HitRec* hits, uint32_t path0, uint32_t npix, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t value, uint32_t n, hipStream_t s);

}  // namespace bipt
