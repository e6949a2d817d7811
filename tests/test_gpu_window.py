"""GPU tests of the windowed traversals at the sizes where its pooled
tests, its long lists and its choice of lanes per ray change path.  Bar:
bit-exact to the oracle, counters included, under every schedule."""
import contextlib

import numpy as np
import pytest

import grt
import pyoracle as orc
from conftest import rng
from test_gpu_grid2 import _built, check_levels, check_trace2
from test_gpu_parity import assert_same, check_any, check_closest, check_grid, _random_rays

pytestmark = pytest.mark.gpu


def _soup(n, seed, size=0.2):
    """n random triangles in the unit box."""
    r = rng(seed)
    c = r.random((n, 1, 3)).astype(np.float32)
    return (c + (r.random((n, 3, 3)).astype(np.float32) - np.float32(0.5)) * np.float32(size)
            ).reshape(n, 9)


def _check_plain(sc, rb, o, oa):
    """Traces without counters against the oracle's results."""
    import torch
    hb = grt.HitBatch.empty(rb.n)
    occ = torch.full((rb.n,), 9, dtype=torch.uint8, device="cuda:0")
    sc.trace_closest(rb, hb)
    sc.trace_any(rb, occ)
    g = hb.numpy()
    for k in ("id", "t", "u", "v"):
        assert_same(g[k], o[k], f"hit.{k}")
    assert_same(occ.cpu().numpy(), oa["occluded"], "occluded")


# One cell that lists every triangle: rounds of 64 and 128 pooled tests with
# their remainders, and both sides of the length from which a list is tested
# on its own (192).
@pytest.mark.parametrize("refs", [1, 2, 63, 64, 65, 127, 128, 129, 191, 192, 193, 1000])
def test_one_cell_lists(gpu_ctx, refs):
    v = _soup(refs, refs)
    sc, fr, offs, orefs = check_grid(gpu_ctx, v, np.zeros_like(v), 1e-5)
    assert len(offs) == 2 and len(orefs) == refs
    for n in (1, 63, 64, 65, 513):
        rays = _random_rays(n, 100 + n)
        check_closest(sc, fr, offs, orefs, v, rays)
        check_any(sc, fr, offs, orefs, v, rays)


# Short and long lists in the same windows, whole and ragged images.
@pytest.mark.parametrize("lam,width", [(0.05, 0), (0.5, 0), (5.0, 37), (60.0, 128)])
def test_mixed_lists(gpu_ctx, lam, width):
    v = np.concatenate([_soup(3000, 7, 0.05), _soup(600, 8, 0.02) * np.float32(0.1) +
                        np.float32(0.4)])
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), lam)
    cam = grt.camera_lookat((0.5, 0.5, -1.5), (0.5, 0.5, 0.0), (0, 1, 0), 60.0, max(width, 61),
                            67)
    rays = orc.primary_rays(grt.camera_dict(cam)) if width else _random_rays(4099, 9)
    check_closest(sc, fr, offs, refs, v, rays, width)
    check_any(sc, fr, offs, refs, v, rays)


# The same on two levels, with lists of both kinds (top cells, sub-cells) on
# both sides of the length from which the wave tests a list on its own.
@pytest.mark.parametrize("n", [31_999, 32_000, 149_999, 150_000, 299_999, 300_000, 999_999,
                               1_000_000])
def test_two_level_lanes_by_launch_size(gpu_ctx, n):
    v = np.concatenate([_soup(230, 3, 1.2), _soup(400, 4, 0.02) * np.float32(0.1) +
                        np.float32(0.45)])
    sc = _built(gpu_ctx, v, np.zeros_like(v), 0.2, 0.1, 250)
    fr, offs, refs, g2 = check_levels(sc, v, 0.2, 0.1, 250)
    lens, sub = np.diff(offs), np.diff(g2[1])
    plain = lens[(lens > 0) & (lens < 250)]
    assert plain.max() >= 192 and plain.min() < 192 and sub.max() >= 192 and sub.min() < 192
    rays = _random_rays(n, 5)
    check_trace2(sc, fr, offs, refs, g2, v, rays, one_level=False, modes=[("simple", 16)])
    _check_plain(sc, grt.RayBatch.from_numpy(rays),
                 orc.grid2_trace_closest(fr, offs, refs, g2, v, rays),
                 orc.grid2_trace_any(fr, offs, refs, g2, v, rays))


# Both sides of the size up to which a fixed number of lanes per ray holds.
@pytest.mark.parametrize("n", [499_999, 500_000])
def test_two_level_fixed_lanes(gpu_ctx, n):
    v = np.concatenate([_soup(230, 3, 1.2), _soup(400, 4, 0.02) * np.float32(0.1) +
                        np.float32(0.45)])
    sc = _built(gpu_ctx, v, np.zeros_like(v), 0.2, 0.1, 250)
    fr, offs, refs, g2 = check_levels(sc, v, 0.2, 0.1, 250)
    check_trace2(sc, fr, offs, refs, g2, v, _random_rays(n, 5), one_level=False,
                 modes=[("split", k) for k in (2, 4, 8, 16)])
    rb = grt.RayBatch.from_numpy(_random_rays(n, 5))
    o, oa = (f(fr, offs, refs, g2, v, _random_rays(n, 5))
             for f in (orc.grid2_trace_closest, orc.grid2_trace_any))
    for k in (2, 4, 8, 16):
        gpu_ctx.set_trace_mode("split", k)
        _check_plain(sc, rb, o, oa)
    gpu_ctx.set_trace_mode("simple", 16)


# Both sides of every size at which the lanes per ray change.
@pytest.mark.parametrize("n", [99_999, 100_000, 399_999, 400_000, (4 << 20) - 1, 4 << 20])
def test_lanes_by_launch_size(gpu_ctx, n):
    import torch
    v = _soup(64, 3, 0.4)
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), 4.0)
    rays = _random_rays(n, 5)
    o = orc.trace_closest(fr, offs, refs, v, rays, counters=True)
    oa = orc.trace_any(fr, offs, refs, v, rays, counters=True)
    rb, hb = grt.RayBatch.from_numpy(rays), grt.HitBatch.empty(n)
    occ = torch.full((n,), 9, dtype=torch.uint8, device="cuda:0")
    cnt = torch.full((2 * n,), -7, dtype=torch.int32, device="cuda:0")
    gpu_ctx.set_trace_mode("simple", 16)
    for counters in (cnt, None):
        sc.trace_closest(rb, hb, counters=counters)
        g = hb.numpy()
        for k in ("id", "t", "u", "v"):
            assert_same(g[k], o[k], f"hit.{k}")
        if counters is not None:
            c = cnt.cpu().numpy().view(np.uint32).reshape(n, 2)
            assert_same(c[:, 0], o["cells"], "cells visited")
            assert_same(c[:, 1], o["tests"], "triangle tests")
        sc.trace_any(rb, occ, counters=counters)
        assert_same(occ.cpu().numpy(), oa["occluded"], "occluded")
        if counters is not None:
            c = cnt.cpu().numpy().view(np.uint32).reshape(n, 2)
            assert_same(c[:, 0], oa["cells"], "cells visited")
            assert_same(c[:, 1], oa["tests"], "triangle tests")


# Flat grids take other lanes per ray: both sides of every size at which these
# change, with the flat grid known to the host, and not known (no build, no
# check since the reservation), where the launch goes by its size alone.
@pytest.mark.parametrize("n", [99_999, 100_000, 399_999, 400_000, 999_999, 1_000_000,
                               (4 << 20) - 1, 4 << 20])
def test_flat_lanes_by_launch_size(gpu_ctx, n):
    import torch
    v = (_soup(64, 3, 0.4).reshape(-1, 3) * np.float32([1.0, 0.04, 1.0])).reshape(-1, 9)
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), 4.0)
    cells = fr["n"][0] * fr["n"][1] * fr["n"][2]
    assert (max(fr["n"]) / 2.5) ** 3 >= cells
    rays = _random_rays(n, 5)
    o = orc.trace_closest(fr, offs, refs, v, rays, counters=True)
    oa = orc.trace_any(fr, offs, refs, v, rays, counters=True)
    rb, hb = grt.RayBatch.from_numpy(rays), grt.HitBatch.empty(n)
    occ = torch.full((n,), 9, dtype=torch.uint8, device="cuda:0")
    cnt = torch.full((2 * n,), -7, dtype=torch.int32, device="cuda:0")
    gpu_ctx.set_trace_mode("simple", 16)
    _check_plain(sc, rb, o, oa)
    for r in (o, oa):
        if r is o:
            sc.trace_closest(rb, hb, counters=cnt)
        else:
            sc.trace_any(rb, occ, counters=cnt)
        c = cnt.cpu().numpy().view(np.uint32).reshape(n, 2)
        assert_same(c[:, 0], r["cells"], "cells visited")
        assert_same(c[:, 1], r["tests"], "triangle tests")
    unchecked = grt.Scene(gpu_ctx)
    unchecked.upload(v, np.zeros_like(v))
    unchecked.reserve_grid(int(cells), len(refs))
    unchecked.rebuild_grid_async(4.0)
    _check_plain(unchecked, rb, o, oa)
    unchecked.close()
    sc.close()


# Waves with few rays to walk give them more lanes: every number of walking
# rays per wave around the powers of two, first, last and scattered in it, on
# one level and two.
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("n", [64 * 40 + 7, 1_000_003])
def test_sparse_waves(gpu_ctx, two, n):
    v = np.concatenate([_soup(300, 3, 0.6), _soup(400, 4, 0.02) * np.float32(0.1) +
                        np.float32(0.45)])
    sc = _built(gpu_ctx, v, np.zeros_like(v), 2.0, 4.0 if two else 0.0, 16)
    rays = _random_rays(n, 11)
    w, l = np.arange(n) // 64, np.arange(n) % 64
    k = np.array([1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 0])[w % 16]
    place = np.where(w // 16 % 3 == 0, l, np.where(w // 16 % 3 == 1, 63 - l, l * 37 % 64))
    off = place >= k
    rays["tmin"][off], rays["tmax"][off] = 1.0, -1.0
    if two:
        fr, offs, refs, g2 = check_levels(sc, v, 2.0, 4.0, 16)
        check_trace2(sc, fr, offs, refs, g2, v, rays, one_level=False,
                     modes=[("simple", 16), ("split", 2), ("split", 8)])
        _check_plain(sc, grt.RayBatch.from_numpy(rays),
                     orc.grid2_trace_closest(fr, offs, refs, g2, v, rays),
                     orc.grid2_trace_any(fr, offs, refs, g2, v, rays))
        return
    _, offs, refs = sc.download_grid()
    fr = orc.grid_frame(v, 2.0)
    check_closest(sc, fr, offs, refs, v, rays)
    check_any(sc, fr, offs, refs, v, rays)
    _check_plain(sc, grt.RayBatch.from_numpy(rays), orc.trace_closest(fr, offs, refs, v, rays),
                 orc.trace_any(fr, offs, refs, v, rays))


# An uploaded cell may list triangles again and again, past the 28 bits of a
# window key's position: the nearest record decides also there, of two at the
# same t the first, and an any-hit ray stops at the first occluder.
def test_list_longer_than_a_key_position(gpu_ctx):
    import torch
    sec, n = 1 << 28, (1 << 28) + 300
    tri = lambda x, z: [x, 0.1, z, x + 0.15, 0.1, z, x, 0.9, z]
    v = np.array([[0.97, 0.97, 0.97, 0.98, 0.97, 0.97, 0.97, 0.98, 0.97],   # 0: in no ray's way
                  tri(0.0, 0.5), tri(0.0, 0.3), tri(0.25, 0.4), tri(0.25, 0.4),
                  tri(0.5, 0.5), tri(0.75, 0.6), tri(0.75, 0.2)], np.float32)
    fr = orc.grid_frame(v, 1e-6)
    assert list(fr["n"]) == [1, 1, 1]
    refs = np.zeros(n, np.uint32)
    refs[100], refs[sec + 5] = 1, 2       # the nearer one in the second 2^28
    refs[200], refs[sec + 7] = 3, 4       # the same t in both: the first
    refs[sec + 131] = 5                   # only there
    refs[9], refs[sec + 9] = 6, 7         # at the same position modulo 2^28
    offs = np.array([0, n], np.uint32)
    at = [0, 8, 16, 24]                   # each in a wave of its own
    rays = {k: np.zeros(32, np.float32) for k in ("ox", "oy", "oz", "dx", "dy", "dz")}
    rays.update(tmin=np.ones(32, np.float32), tmax=-np.ones(32, np.float32))
    rays["ox"][at] = [0.02, 0.27, 0.52, 0.77]
    rays["oy"][:], rays["oz"][:], rays["dz"][:] = 0.2, -1.0, 1.0
    rays["tmin"][at], rays["tmax"][at] = 0.0, np.inf
    sc = grt.Scene(gpu_ctx)
    sc.upload(v, np.zeros_like(v))
    sc.upload_grid(fr, offs, refs)
    gpu_ctx.set_trace_mode("simple", 16)
    rb, hb = grt.RayBatch.from_numpy(rays), grt.HitBatch.empty(32)
    sc.trace_closest(rb, hb)
    # triangle 0 is never hit: the oracle walks the others alone, in their order
    few = refs[refs != 0]
    foffs = np.array([0, len(few)], np.uint32)
    g, o = hb.numpy(), orc.trace_closest(fr, foffs, few, v, rays)
    assert list(o["id"][at]) == [2, 3, 5, 7]
    for k in ("id", "t", "u", "v"):
        assert_same(g[k], o[k], f"hit.{k}")
    # in a batch; all four in one wave, with counters
    hb = grt.HitBatch.empty(32)
    with contextlib.closing(grt.Batch(gpu_ctx, 1)) as batch:
        batch.set([(sc, rb, hb, None, 0)])
        batch.trace()
    for k in ("id", "t", "u", "v"):
        assert_same(hb.numpy()[k], o[k], f"hit.{k}")
    cnt = torch.full((64,), -7, dtype=torch.int32, device="cuda:0")
    hb = grt.HitBatch.empty(32)
    gpu_ctx.set_trace_mode("split", 2)
    sc.trace_closest(rb, hb, counters=cnt)
    gpu_ctx.set_trace_mode("simple", 16)
    for k in ("id", "t", "u", "v"):
        assert_same(hb.numpy()[k], o[k], f"hit.{k}")
    c = cnt.cpu().numpy().view(np.uint32).reshape(32, 2)
    assert list(c[at, 0]) == [1] * 4 and list(c[at, 1]) == [n] * 4
    occ = torch.full((32,), 9, dtype=torch.uint8, device="cuda:0")
    cnt = torch.full((64,), -7, dtype=torch.int32, device="cuda:0")
    sc.trace_any(rb, occ, counters=cnt)
    oa = orc.trace_any(fr, foffs, few, v, rays, counters=True)
    assert list(few[oa["tests"][at] - 1]) == [1, 3, 5, 6]
    oa["tests"][at] = [101, 201, sec + 132, 10]
    assert_same(occ.cpu().numpy(), oa["occluded"], "occluded")
    c = cnt.cpu().numpy().view(np.uint32).reshape(32, 2)
    assert_same(c[:, 0], oa["cells"], "cells visited")
    assert_same(c[:, 1], oa["tests"], "triangle tests")
    sc.close()
