"""Queues of the wavefront loop at image sizes that do not fill their 8x8
tiles: every pixel is rendered once per sample, whatever the pass size.

The reference value is the same render in other passes (a path's samples do
not depend on the pass it runs in, so the images are equal bit for bit) and
the oracle under the same per-path streams.
"""
import numpy as np
import pytest

from lajolla_public_amd import api, scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (7, 5), (8, 8), (9, 8), (8, 9), (17, 3), (65, 33)]


@pytest.mark.parametrize("w,h", SIZES)
def test_ragged_image_in_any_pass(w, h):
    desc = scenes.cornell_box(seed=2, width=w, height=h, spp=3, max_depth=4)
    sc = api.Scene(desc)
    img, st = sc.render(stats=True)
    assert st["camera_paths"] == 3 * w * h
    for cap in (64, 192, 1000):
        part, sp = sc.render(options=scenes.render_options(**desc.options),
                             exec_options=api.exec_options(max_paths_in_flight=cap), stats=True)
        assert np.array_equal(img, part), (w, h, cap)
        assert (sp["extension_rays"], sp["shadow_rays"]) == (st["extension_rays"], st["shadow_rays"])
    ref, _ = po.OracleScene(desc).render(plan=1)
    diff = np.abs(img.astype(np.float64) - ref)
    # one sample's FP32 path state against FP64: a path that parts at an edge changes its pixel
    assert (diff <= 1e-3 * np.abs(ref) + 1e-4).all(axis=2).mean() >= (0.95 if w * h > 40 else 0.85)


@pytest.mark.parametrize("cap", [64, 100, 1 << 12])
def test_ragged_batch_in_any_pass(cap):
    """Jobs whose work starts and ends inside a pass and inside a tile."""
    desc = scenes.cornell_box(seed=2, width=16, height=16, spp=2, max_depth=4)
    sc = api.Scene(desc)
    rng = np.random.default_rng(4)
    jobs = [dict(scene=sc, camera=scenes.orbit_camera(desc, rng, w, h, yaw_deg=3, pitch_deg=1, dist_range=(1, 1)), spp=s,
                 max_depth=4, seed=11 + k) for k, (w, h, s) in enumerate([(9, 7, 2), (1, 1, 5), (24, 8, 1), (13, 21, 3)])]
    imgs, _, st = api.render_batch(jobs, api.exec_options(max_paths_in_flight=cap))
    assert st["samples"] == sum(j["camera"]["width"] * j["camera"]["height"] * j["spp"] for j in jobs)
    for j, img in zip(jobs, imgs):
        import copy
        d = copy.copy(desc)
        d.camera = j["camera"]
        one = api.Scene(d).render(samples_per_pixel=j["spp"], max_depth=4, seed=j["seed"])
        # the same samples, added in another order in FP64 and rounded once to FP32
        assert np.allclose(img, one, rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("w,h,spp", [(31, 33, 1), (64, 16, 1), (64, 64, 1), (64, 65, 2), (320, 257, 1), (640, 480, 2)])
def test_material_sort_at_block_edges(w, h, spp):
    """Several material types and misses, queues from under one wave's 1,024 entries to past the traversal's first
    tickets: the image does not depend on the traversal grid (who takes which chunk) nor on the pass."""
    desc = scenes.textured_showcase(seed=5)
    desc.camera = scenes.orbit_camera(desc, np.random.default_rng(3), w, h, yaw_deg=4, pitch_deg=2, dist_range=(1, 1))
    desc.options.update(samples_per_pixel=spp, max_depth=5)
    sc = api.Scene(desc)
    img, st = sc.render(stats=True)
    assert np.isfinite(img).all() and img.mean() > 0
    for bpc, cap in ((1, 0), (3, 0), (8, 1 << 12), (1, 1000)):
        if cap and w * h * spp > 100000:
            continue
        got, sg = sc.render(options=scenes.render_options(**desc.options), stats=True,
                            exec_options=api.exec_options(max_paths_in_flight=cap, trace_blocks_per_cu=bpc))
        assert (sg["extension_rays"], sg["shadow_rays"]) == (st["extension_rays"], st["shadow_rays"])
        if cap == 0:
            assert np.array_equal(img, got), (bpc, cap)
        else:  # a pixel's samples added in other groups in FP64, rounded once to FP32
            assert np.allclose(img, got, rtol=2e-6, atol=1e-9), (bpc, cap)
