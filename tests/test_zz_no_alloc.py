"""bi_pt_trace_closest_noalloc: closest-hit queries that allocate and build nothing.  Its results
equal the restatement's traversal, and bi_pt_trace_closest's, bit for bit, on the box-room
scene and on a scene without triangles; sizes beyond the maximum and a scene whose LBVH is
not current are refused.  Queries of one context share nothing but the scene: those that overlap
on two streams return what each returns alone."""
import ctypes as C

import numpy as np
import pytest

import bi_pt
import scenes

pytestmark = pytest.mark.gpu


def random_rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform((-5.5, 0.2, -5.5), (5.5, 3.8, 5.5), (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    return o, d


def assert_same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))


def oracle_hits(ora, o, d, tmax):
    """(t, triangle, u, v) of the restatement, laid out as bi_pt_trace_closest returns them."""
    rec = np.zeros((len(o), 8), np.float32)
    rec[:, 0:3], rec[:, 3], rec[:, 4:7], rec[:, 7] = o, 0.001, d, tmax
    t, leaf, u, v = ora.trace(rec)
    hit = leaf != 0xFFFFFFFF
    tri = np.where(hit, ora.bvh()["order"][np.where(hit, leaf, 0)], 0xFFFFFFFF).astype(np.uint32)
    return np.where(hit, t, np.inf).astype(np.float32), tri, np.where(hit, u, 0).astype(np.float32), np.where(hit, v, 0).astype(np.float32)


def test_noalloc_equals_oracle_and_allocating_query(c0_scene, c0_oracle):
    print("case: noalloc closest hits vs the oracle and bi_pt_trace_closest, c0, 200000 then 70001 rays", flush=True)
    t = bi_pt.PathTracer()
    t.set_scene(c0_scene)
    with pytest.raises(bi_pt.PtError) as e:   # nothing built yet: refused, nothing allocated
        t.trace_closest_noalloc(*random_rays(8, 1))
    assert e.value.status == 6
    t.render(scenes.camera_c0(16, 16), spp=1, max_bounces=3, seed=1)   # builds the LBVH
    for n, seed in ((200000, 2), (70001, 3)):
        o, d = random_rays(n, seed)
        want = t.trace_closest(o, d, tmax=1000.0)
        got = t.trace_closest_noalloc(o, d, tmax=1000.0)
        assert_same(got, want)
        assert_same(got, oracle_hits(c0_oracle, o, d, 1000.0))
        hits = int((want[1] != 0xFFFFFFFF).sum())
        print(f"{n} rays: {hits} hits, equal", flush=True)
        assert 0 < hits < n
    # a shorter extent, then the maximum size
    o, d = random_rays(bi_pt.NOALLOC_MAX_RAYS, 4)
    got = t.trace_closest_noalloc(o, d, tmax=2.5)
    assert_same(got, t.trace_closest(o, d, tmax=2.5))
    assert_same(got, oracle_hits(c0_oracle, o, d, 2.5))
    with pytest.raises(bi_pt.PtError) as e:
        t.trace_closest_noalloc(*random_rays(bi_pt.NOALLOC_MAX_RAYS + 1, 5))
    assert e.value.status == 1
    # a changed scene is refused until it is built again
    t.update_transforms(c0_scene.instances["xform"])
    with pytest.raises(bi_pt.PtError) as e:
        t.trace_closest_noalloc(*random_rays(8, 6))
    assert e.value.status == 6
    o, d = random_rays(5000, 7)
    want = t.trace_closest(o, d)          # builds again
    assert_same(t.trace_closest_noalloc(o, d), want)
    t.stats()                             # no device error flag
    t.close()


def test_noalloc_scene_without_triangles():
    print("case: noalloc closest hits on a scene without triangles", flush=True)
    sky, col = scenes.constant_sky()
    empty = scenes.Scene("empty", [], np.zeros(0, scenes.INSTANCE_DTYPE),
                         scenes.material((0.5, 0.5, 0.5), 0.5, 0.0)[None],
                         scenes.dir_light((1, 1, 1), (0, 1, 0))[None], sky, col, np.eye(3, dtype=np.float32).reshape(-1))
    t = bi_pt.PathTracer()
    t.set_scene(empty)
    t.render(scenes.camera_c0(8, 8), spp=1, max_bounces=3, seed=1)
    for n in (3000, 17):
        o, d = random_rays(n, n)
        got = t.trace_closest_noalloc(o, d)
        assert np.all(np.isinf(got[0])) and np.all(got[1] == 0xFFFFFFFF)
        assert_same(got, t.trace_closest(o, d))
    t.close()


def test_queries_overlap_on_two_streams(c0_scene, c0_oracle):
    """Closest-hit queries (both entry points) and occlusion queries of one context, enqueued in
    turn on two streams without a wait between them."""
    import torch
    print("case: c0, overlapping queries on two streams, 150000 / 90001 / 120000 rays", flush=True)
    t = bi_pt.PathTracer()
    t.set_scene(c0_scene)
    t.trace_closest(*random_rays(8, 1))   # builds, and waits for it
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    calls = []
    for k, (entry, n, tmax) in enumerate([("closest", 150000, 1000.0), ("noalloc", 90001, 1000.0), ("occlusion", 120000, 3.0)] * 4):
        o, d = random_rays(n, 50 + k % 3)
        cols, rays, dev = t._query_rays(o, d)
        f32 = dict(dtype=torch.float32, device=dev)
        out = [torch.full((n,), -1.0, **f32), torch.full((n,), 7, dtype=torch.int32, device=dev),
               torch.full((n,), -1.0, **f32), torch.full((n,), -1.0, **f32)]
        calls.append((entry, n, tmax, o, d, cols, rays, out))
    torch.cuda.synchronize()
    p = lambda x: C.c_void_p(x.data_ptr())   # noqa: E731
    lib = bi_pt.lib()
    for k, (entry, n, tmax, _, _, _, rays, out) in enumerate(calls):
        s = C.c_void_p(streams[(k + k // 3) % 2].cuda_stream)
        if entry == "occlusion":
            st = lib.bi_pt_trace_occlusion(t.h, n, C.byref(rays), tmax, p(out[1]), s)
        else:
            fn = lib.bi_pt_trace_closest if entry == "closest" else lib.bi_pt_trace_closest_noalloc
            st = fn(t.h, n, C.byref(rays), tmax, p(out[0]), p(out[1]), p(out[2]), p(out[3]), s)
        assert st == 0
    torch.cuda.synchronize()
    want = {}
    for entry, n, tmax, o, d, _, _, out in calls:
        if entry not in want:
            if entry == "occlusion":
                rec = np.zeros((n, 8), np.float32)
                rec[:, 0:3], rec[:, 3], rec[:, 4:7], rec[:, 7] = o, 0.001, d, tmax
                want[entry] = (c0_oracle.trace(rec, any_hit=True)[0],)
            else:
                want[entry] = oracle_hits(c0_oracle, o, d, tmax)
        got = (out[1],) if entry == "occlusion" else (out[0], out[1], out[2], out[3])
        assert_same([g.cpu().numpy() for g in got], want[entry])
    t.stats()
    t.close()
