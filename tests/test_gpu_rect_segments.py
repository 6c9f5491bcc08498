"""The rect lights' kernel runs after each segment's shading and owns its slot: paths that end
in the radiance cache or restart at it (training paths), misses, the folded quadrants of the
tables' azimuth and clipped quads, and waves whose jobs differ in size and in having rect
lights, against the oracle."""
import numpy as np
import pytest

import bi_pt
import scenes
from test_gpu_nrc import constant_params
from test_gpu_parity import radiance_check
from test_gpu_rect_lights import rect_c0

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bounce", [1, 3])
def test_cached_paths_with_rect_lights(oracle_lib, bounce):
    """The constant cache's image and the training records equal the restatement's; targets
    are sums of the slots, in one order, so they are equal too."""
    print(f"case: c0 + rect lights 53x37, cache at segment {bounce}", flush=True)
    sc, cam, k = rect_c0(), scenes.camera_c0(53, 37), np.array([0.5, 0.25, 0.125], np.float32)
    ora = oracle_lib.OracleScene(sc)
    t = bi_pt.PathTracer()
    t.set_scene(sc)
    nrc = bi_pt.Nrc(t, train_samples=4096, train_steps=4, cache_bounce=bounce)
    nrc.set_params(constant_params(k))
    nrc.render(cam, spp=2, max_bounces=5, seed=77)
    assert radiance_check(t.sums(cam.width * cam.height), ora.render32_cached(cam, 5, 77, 2, bounce, k))
    nrc.render(cam, spp=1, max_bounces=5, seed=5)
    rec, tgt = nrc.samples(4096)
    orec, otgt = ora.train_samples(cam, 5, bi_pt.nrc_train_seed(5, 1), bounce, 4096)
    assert np.array_equal(rec.view(np.uint32), orec.view(np.uint32))
    assert np.array_equal(tgt.view(np.uint32), otgt.view(np.uint32))
    nrc.close()
    t.close()


@pytest.mark.parametrize("sizes", [((1, 1), (17, 3)), ((64, 4), (63, 5), (257, 1))])
@pytest.mark.parametrize("one_light", [False, True])
def test_mixed_waves(oracle_lib, sizes, one_light):
    print(f"case: batch of c0 with / without rect lights at {sizes}", flush=True)
    b = bi_pt.Batch()
    jobs, want = [], []
    for k, (w, h) in enumerate(sizes):
        sc = scenes.scene_c0() if k == 1 else rect_c0(seed=k)
        if one_light and k != 1:
            sc.rect_lights = sc.rect_lights[1:]
        cam = scenes.camera_c0(w, h)
        t = bi_pt.PathTracer()
        t.set_scene(sc)
        jobs.append((t, bi_pt.Job(t, cam, spp=3, max_bounces=4, seed=9 + k)))
        want.append(oracle_lib.OracleScene(sc).render32(cam, 4, 9 + k, spp=3)["sums"])
    b.render([j for _, j in jobs])
    ok = [radiance_check(t.sums(w * h), x) for (t, _), (w, h), x in zip(jobs, sizes, want)]
    for t, _ in jobs:
        t.close()
    b.close()
    assert all(ok)


def test_graph_follows_rect_lights(oracle_lib):
    """A replayed batch whose second job gains, keeps and loses rect lights while no buffer
    changes (the first job's three lights already give every path a slot more than the second
    job uses): each call equals the oracle's image of the scene as it then is."""
    import torch
    print("case: graph batch of c0 with three suns and c0, rect lights set and unset on the second", flush=True)
    suns = scenes.scene_c0()
    suns.dir_lights = np.stack([scenes.dir_light((0.9, 0.8, 0.7), d) for d in ((0.3, 0.8, 0.4), (-0.4, 0.7, 0.2), (0.1, 0.9, -0.5))])
    plain, rect = scenes.scene_c0(), rect_c0(seed=2)
    cam = scenes.camera_c0(40, 24)
    ts = []
    for sc in (suns, rect):
        t = bi_pt.PathTracer()
        t.set_scene(sc)
        ts.append(t)
    ts[1].set_rect_lights(None)
    b = bi_pt.Batch()
    b.set_tuning(use_graph=True)
    stream = torch.cuda.Stream()
    want = {k: oracle_lib.OracleScene(sc).render32(cam, 4, 21, spp=2)["sums"]
            for k, sc in (("suns", suns), ("plain", plain), ("rect", rect))}
    ok = []
    for lights in (None, None, rect.rect_lights, rect.rect_lights, None):
        ts[1].set_rect_lights(lights)
        b.render([bi_pt.Job(t, cam, spp=2, max_bounces=4, seed=21) for t in ts], stream=stream.cuda_stream)
        stream.synchronize()
        got = [t.sums(cam.width * cam.height) for t in ts]
        torch.cuda.synchronize()
        ok += [radiance_check(got[0], want["suns"]), radiance_check(got[1], want["rect" if lights is not None else "plain"])]
    for t in ts:
        t.close()
    b.close()
    assert all(ok), ok
