"""Closest-hit and occlusion queries on trees and rays at the edges of the traversal's node
format, against the restatement, bit for bit: trees of one to a few nodes, scenes far from
the origin and of extreme size, rays along an axis, from a face, and rays that are no
numbers; query sizes around a wavefront, a workgroup and more than the chip holds at once."""
import dataclasses

import numpy as np
import pytest

import bi_pt
import scenes

pytestmark = pytest.mark.gpu


def moved(scene, scale, shift):
    s = dataclasses.replace(scene, instances=scene.instances.copy())
    x = s.instances["xform"].reshape(-1, 3, 4)
    x *= np.float32(scale)
    x[:, :, 3] += np.float32(shift)
    return s


def edge_rays(rng, n, scale, shift):
    o = rng.uniform(-7.0, 7.0, (n, 3)) * scale + shift
    d = rng.uniform(-6.0, 6.0, (n, 3)) * scale + shift - o
    d = d / np.linalg.norm(d, axis=1, keepdims=True)
    k = rng.integers(0, 3, n)
    axis = rng.random(n) < 0.2                      # along an axis, both signs of zero elsewhere
    d[axis] = rng.choice([0.0, -0.0], (int(axis.sum()), 3))
    d[axis, k[axis]] = rng.choice([-1.0, 1.0], int(axis.sum()))
    o = np.where(rng.random((n, 3)) < 0.1, np.round(o), o)
    bad = rng.random(n)
    o[bad < 0.01, 0] = np.nan
    d[(bad > 0.01) & (bad < 0.02), 1] = np.nan
    o[(bad > 0.02) & (bad < 0.03), 2] = np.inf
    d[(bad > 0.03) & (bad < 0.04), 0] = -np.inf
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("tris,rays,scale,shift", [
    (1, 64, 1.0, 0.0), (2, 65, 1.0, 0.0), (3, 1, 1.0, 0.0), (5, 257, 1.0, 0.0), (8, 63, 1.0, 0.0), (300, 20000, 1.0, 0.0),
    (300, 20000, 1.0, 4e4), (300, 20000, 1e6, 0.0), (300, 20000, 1e11, 3e12), (4000, 70001, 1.0, 100.0), (40, 600001, 1.0, 0.0),
])
def test_queries_match_restatement(oracle_lib, tris, rays, scale, shift):
    print(f"case: {tris} triangles x {scale:g} + {shift:g}, {rays} rays", flush=True)
    sc = moved(scenes.scene_random_triangles(tris, 5), scale, shift)
    rng = np.random.default_rng(tris + rays)
    o, d = edge_rays(rng, rays, scale, shift)
    tmax = 1000.0 * max(scale, 1.0)
    ref = oracle_lib.OracleScene(sc)
    rec = np.zeros((rays, 8), np.float32)
    rec[:, 0:3], rec[:, 3], rec[:, 4:7], rec[:, 7] = o, 0.001, d, tmax
    ot, oleaf, ou, ov = ref.trace(rec)
    hit = oleaf != 0xFFFFFFFF
    order = ref.bvh()["order"]
    g = bi_pt.PathTracer()
    g.set_scene(sc)
    t, tri, u, v = g.trace_closest(o, d, tmax=tmax)
    assert np.array_equal(tri != 0xFFFFFFFF, hit)
    assert np.array_equal(tri[hit], order[oleaf[hit]])
    for a, b in ((t, ot), (u, ou), (v, ov)):
        assert np.array_equal(a[hit].view(np.uint32), b[hit].view(np.uint32))
    assert np.all(np.isinf(t[~hit])) and np.all(u[~hit] == 0) and np.all(v[~hit] == 0)
    assert np.array_equal(g.trace_occlusion(o, d, tmax=tmax), ref.trace(rec, any_hit=True)[0])
    g.close()
