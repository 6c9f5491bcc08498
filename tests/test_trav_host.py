"""The traversal's compressed nodes and visit test, compiled for the CPU, against the exact
slab test.

`bisemutum-engine_amd/csrc/pt_trav.hpp` packs a node's child boxes to 8-bit planes and tests
them with fused multiply-adds; the result only decides which nodes a ray visits.  Hits stay
those of the exact FP32 test if and only if the visit test never skips a box that the exact
test passes, which `tests/host_wave/trav_host.cpp` counts over boxes and rays of every kind
that could break it: boxes of any size and distance, flat and single-point boxes, boxes of very
different size in one node, rays along an axis, from a face or a corner, through corners, with
zero direction components, at coordinates up to the range's end, and boxes that are no numbers.
A ray whose origin times inverse direction overflows (an origin that is infinite, or far
away along an axis that the direction does not follow) must not walk the tree either: the exact
test rejects it at the root, and the visit test has to as well.
"""
import functools
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REC = np.dtype([("box", np.float32, (4, 6)), ("n", np.int32), ("o", np.float32, 3), ("d", np.float32, 3),
                ("tmax", np.float32)])


@pytest.fixture(scope="module")
def host_binary(tmp_path_factory):
    exe = tmp_path_factory.mktemp("trav") / "trav_host"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wall", "-Wextra", "-Wno-unknown-pragmas", "-o",
                    str(exe), os.path.join(HERE, "host_wave", "trav_host.cpp")], check=True)
    return exe


def records(n, rng, centre=0.0, spread=4.0, size=1.0, size_decades=2.0, origin_spread=8.0):
    r = np.zeros(n, REC)
    c = centre + rng.uniform(-spread, spread, (n, 1, 3)) + rng.uniform(-1, 1, (n, 4, 3)) * size
    half = size * 10.0 ** -rng.uniform(0, size_decades, (n, 4, 3)) * 0.5
    r["box"][..., :3] = c - half
    r["box"][..., 3:] = np.maximum(c + half, r["box"][..., :3].astype(np.float64))
    r["n"] = rng.integers(1, 5, n)
    r["o"] = centre + rng.uniform(-origin_spread, origin_spread, (n, 3))
    aim(r, rng, c[:, 0] + rng.uniform(-1.5, 1.5, (n, 3)) * half[:, 0])
    r["tmax"] = np.where(rng.random(n) < 0.3, 10.0 ** rng.uniform(-2, 2, n), 1000.0)
    return r


def aim(r, rng, target):
    d = target - r["o"].astype(np.float64)
    r["d"] = d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-300)


@functools.lru_cache(maxsize=None)
def families():
    rng = np.random.default_rng(11)
    n = 40000
    out = {"ordinary": records(n, rng)}
    out["tiny, far from the origin"] = records(n, rng, centre=1e4, spread=1.0, size=1e-3, origin_spread=50.0)
    out["tiny at unit coordinates"] = records(n, rng, centre=3.0, spread=0.1, size=1e-6, origin_spread=2.0)
    out["one large, others tiny"] = records(n, rng, size_decades=7.0)
    out["large coordinates"] = records(n, rng, centre=0.0, spread=1e8, size=1e7, origin_spread=3e8)
    out["large coordinates"]["tmax"] = 1.7e38
    flat = records(n, rng)
    for a in range(3):
        m = rng.random(n) < 0.5
        flat["box"][m, :, 3 + a] = flat["box"][m, :, a]
    out["flat"] = flat
    grid = records(n, rng)   # tie-rich: integer boxes, origins and directions
    grid["box"] = np.round(grid["box"])
    grid["box"][..., 3:] = np.maximum(grid["box"][..., 3:], grid["box"][..., :3])
    grid["o"] = np.round(grid["o"])
    grid["d"] = rng.integers(-2, 3, (n, 3))
    out["integers"] = grid
    corner = records(n, rng)   # through a corner of the first box, in FP32
    pick = rng.integers(0, 2, (n, 3)).astype(bool)
    aim(corner, rng, np.where(pick, corner["box"][:, 0, 3:], corner["box"][:, 0, :3]).astype(np.float64))
    out["through corners"] = corner
    axis = records(n, rng)
    a = rng.integers(0, 3, n)
    d = np.zeros((n, 3))
    d[np.arange(n), a] = rng.choice([-1.0, 1.0, 1e-3, -1e-18], n)
    axis["d"] = d
    on = rng.random((n, 3)) < 0.4   # on a face's plane
    axis["o"] = np.where(on, np.where(pick, axis["box"][:, 0, 3:], axis["box"][:, 0, :3]), axis["o"])
    out["along an axis"] = axis
    face = records(n, rng)   # starting on a face, leaving
    w = rng.random((n, 3))
    p = face["box"][:, 1, :3] * (1 - w) + face["box"][:, 1, 3:] * w
    k = rng.integers(0, 3, n)
    p[np.arange(n), k] = np.where(pick[:, 0], face["box"][np.arange(n), 1, 3 + k], face["box"][np.arange(n), 1, k])
    face["o"] = p
    out["from a face"] = face
    unit = records(n, rng)   # directions of any length
    unit["d"] = unit["d"] * 10.0 ** rng.uniform(-25, 25, (n, 1))
    unit["tmax"] = 1.7e38
    out["directions of any length"] = unit
    huge = records(n, rng, spread=1e20, size=1e19, origin_spread=1e20)
    huge["d"][rng.random((n, 3)) < 0.2] = 0.0
    huge["tmax"] = 1.7e38
    out["huge"] = huge
    end = records(n, rng, spread=1e37, size=1e38, origin_spread=1e37)
    end["tmax"] = 1.7e38
    out["the range's end"] = end
    nan = records(n, rng)
    m = rng.random((n, 4, 6)) < 0.1
    nan["box"][m] = np.nan
    nan["box"][rng.random((n, 4, 6)) < 0.03] = np.inf
    nan["box"][rng.random((n, 4, 6)) < 0.03] = -np.inf
    out["not numbers"] = nan
    zero = records(n, rng, centre=0.0, spread=1e-38, size=1e-39, origin_spread=1.0)
    out["subnormal"] = zero
    return out


@pytest.mark.parametrize("name", sorted(families()))
def test_no_box_is_skipped(host_binary, tmp_path, name):
    r = families()[name]
    src = tmp_path / "in.bin"
    r.tofile(src)
    got = subprocess.run([str(host_binary), str(src)], check=True, capture_output=True, text=True, timeout=120).stdout
    total, hit, skipped, visited, order = map(int, got.split())
    assert total == int(r["n"].sum()) and skipped == 0 and order == 0, (name, total, hit, skipped, visited, order)
    if name in ("ordinary", "flat", "through corners", "large coordinates"):
        assert hit > 0.02 * total
        # planes are rounded by at most two of 252 quanta of the node's extent
        assert visited <= hit * 1.35 + 0.02 * total, (name, hit, visited)


def far_rays(name):
    """Rays that the exact test rejects at any box of ordinary coordinates."""
    rng = np.random.default_rng(29)
    n = 20000
    r = records(n, rng)
    a, rows = rng.integers(0, 3, n), np.arange(n)
    if name == "infinite origin":
        r["o"][rows, a] = rng.choice([-np.inf, np.inf], n)
        more = rng.random((n, 3)) < 0.5
        r["o"][more] = rng.choice([-np.inf, np.inf], int(more.sum()))
        r["d"][rng.random((n, 3)) < 0.2] = 0.0
    else:   # far away on one to three axes, none of which the direction follows except by chance
        far = rng.random((n, 3)) < 0.5
        far[rows, a] = True
        mag = 10.0 ** rng.uniform(20, 38, (n, 3)) * rng.choice([-1.0, 1.0], (n, 3))
        r["o"] = np.where(far, mag, r["o"])
        r["d"] = rng.choice([0.0, -0.0], (n, 3))
        k = (a + rng.integers(1, 3, n)) % 3
        r["d"][rows, k] = rng.choice([-1.0, 1.0], n)
    r["tmax"] = np.where(rng.random(n) < 0.5, 1000.0, 1.7e38)
    return r


@pytest.mark.parametrize("name", ["infinite origin", "far beside the direction"])
def test_far_rays_visit_nothing(host_binary, tmp_path, name):
    r = far_rays(name)
    src = tmp_path / "in.bin"
    r.tofile(src)
    got = subprocess.run([str(host_binary), str(src)], check=True, capture_output=True, text=True, timeout=120).stdout
    total, hit, skipped, visited, order = map(int, got.split())
    assert total == int(r["n"].sum()) and hit == 0 and skipped == 0 and order == 0
    assert visited == 0, (name, visited, total)


def test_large_products_visit_as_the_exact_test(host_binary, tmp_path):
    """Origin times inverse direction between 1e38 and the largest FP32 number: still a
    number, so the axis still rejects what the exact test rejects."""
    rng = np.random.default_rng(31)
    n = 20000
    r = records(n, rng)
    a, rows = rng.integers(0, 3, n), np.arange(n)
    r["o"][rows, a] = rng.uniform(1.1e18, 3.3e18, n) * rng.choice([-1.0, 1.0], n)
    r["d"] = 0.0
    r["d"][rows, (a + 1) % 3] = rng.choice([-1.0, 1.0], n)
    r["tmax"] = 1.7e38
    src = tmp_path / "in.bin"
    r.tofile(src)
    got = subprocess.run([str(host_binary), str(src)], check=True, capture_output=True, text=True, timeout=120).stdout
    total, hit, skipped, visited, order = map(int, got.split())
    assert skipped == 0 and order == 0 and visited <= hit + 0.001 * total, (hit, visited, total)
