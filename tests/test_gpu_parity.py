"""GPU parity: the HIP path against the oracle, called through the C ABI.

* BVH queries: closest-hit primitive ids and distances equal the oracle's
  brute-force-free FP64 BVH (watertight tests on both sides).
* Renders: per-pixel means of the GPU render within the stated statistical
  bound of the oracle's converged FP64 render of the same scene
  (tests/golden/*_oracle.npz, written by tests/golden/make_oracle_images.py).
"""
import os

import numpy as np
import pytest

from naivetrace_amd import abi, configs
from naivetrace_amd.renderer import GpuRenderer

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
pytestmark = pytest.mark.gpu


def _random_rays(n, rng, lo, hi):
    org = rng.uniform(lo, hi, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return org, d


def test_device_info(gpu_lib):
    info = gpu_lib.ttgpu_device_info().decode()
    assert "gfx950" in info


def test_bvh_matches_gpu_bruteforce(gpu_lib):
    """BVH traversal against testing every primitive, both on the device."""
    s = configs.cornell_box(16, 16)
    p = abi.default_params(16, 16)
    rng = np.random.default_rng(4)
    org, d = _random_rays(20000, rng, [-0.95, 0.05, -0.95], [0.95, 1.95, 0.95])
    tmax = np.full(len(org), 1e30)
    with GpuRenderer(s, p) as r:
        t, prim, _, _ = r.trace_closest(org, d, tmax)
        tb, pb, _, _ = r.trace_closest(org, d, tmax, bruteforce=True)
    print("bvh hit rate", np.mean(prim >= 0), "brute-force hit rate", np.mean(pb >= 0), flush=True)
    assert np.array_equal(prim >= 0, pb >= 0)
    # Same triangle test on both sides, so the closest distance agrees (to the last bit where a ray
    # crosses a shared edge).  Where two primitives lie at the same distance -- the boxes' bottom
    # faces are coplanar with the floor -- the BVH's nearest-first order and the brute force's index
    # order may keep different ones.
    np.testing.assert_allclose(t, tb, rtol=3e-7, atol=0)
    differ = prim != pb
    np.testing.assert_allclose(t[differ], tb[differ], rtol=3e-7, atol=0)
    assert np.mean(differ) < 0.005


def test_closest_hit_matches_oracle(gpu_lib, oracle):
    s = configs.cornell_box(16, 16)
    p = abi.default_params(16, 16)
    rng = np.random.default_rng(3)
    org, d = _random_rays(20000, rng, [-0.95, 0.05, -0.95], [0.95, 1.95, 0.95])
    tmax = np.full(len(org), 1e30)
    with GpuRenderer(s, p) as r:
        t, prim, u, v = r.trace_closest(org, d, tmax)
    t_ref, prim_ref = oracle.trace_closest(s, org, d, tmax)
    hit = prim_ref >= 0
    assert hit.mean() > 0.8  # the box is open at the front (z = +1)
    assert np.array_equal(prim >= 0, hit)
    same = prim == prim_ref
    # Primitive ids agree except where two surfaces are hit at the same distance (box bottoms are
    # coplanar with the floor, quads share diagonals); distances agree everywhere (FP32 vs FP64).
    assert same.mean() > 0.97, f"{(~same).sum()} mismatches"
    np.testing.assert_allclose(t[hit], t_ref[hit], rtol=2e-5, atol=2e-6)
    assert np.all((u >= -1e-6) & (v >= -1e-6) & (u + v <= 1 + 1e-5))


def test_closest_hit_empty_and_miss(gpu_lib):
    s = configs.cornell_box(8, 8)
    p = abi.default_params(8, 8)
    with GpuRenderer(s, p) as r:
        t, prim, _, _ = r.trace_closest(np.zeros((0, 3)), np.zeros((0, 3)), np.zeros(0))
        assert len(t) == 0
        # Rays leaving the open front of the box miss everything.
        t, prim, _, _ = r.trace_closest([[0, 1, 5]], [[0, 0, 1]], [1e30])
        assert prim[0] == -1 and np.isinf(t[0])
        # tmax shorter than the wall distance: no hit.
        t, prim, _, _ = r.trace_closest([[0, 1, 0]], [[0, 1, 0]], [0.5])
        assert prim[0] == -1
        occ = r.trace_occluded([[0, 1, 0], [0, 1, 0]], [[0, 1, 0], [0, 1, 0]], [0.5, 3.0])
        assert occ.tolist() == [0, 1]


def _zscores(gpu_mean, gpu_se, ref_mean, ref_se):
    se = np.sqrt(gpu_se ** 2 + ref_se ** 2)
    ok = se > 0
    z = np.zeros_like(gpu_mean)
    z[ok] = (gpu_mean[ok] - ref_mean[ok]) / se[ok]
    # Pixels with zero variance on both sides must agree exactly (up to float rounding).
    assert np.all(np.abs(gpu_mean[~ok] - ref_mean[~ok]) < 1e-6)
    return z


def render_parity(name, mis=abi.MIS_REFERENCE, mode=abi.SAMPLE_BOTH, builder=configs.cornell_box):
    """GPU render of `builder`'s scene against the oracle's render tests/golden/<name>_oracle.npz.

    The GPU renders as many samples per pixel as the fixture holds: per-pixel path estimates are
    right-skewed (rare bright paths), which makes a sample mean and its estimated error correlated;
    with equal sample counts on both sides the z-scores are symmetric and their mean is an unbiased
    check for a systematic difference."""
    f = np.load(os.path.join(GOLDEN, f"{name}_oracle.npz"))
    spp = int(f["spp"])
    w, h, depth = int(f["width"]), int(f["height"]), int(f["max_depth"])
    assert int(f["mis_mode"]) == mis and int(f["sample_mode"]) == mode
    s = builder(w, h)
    p = abi.default_params(w, h, max_depth=depth, seed=11)
    p.mis_mode = mis
    p.sample_mode = mode
    with GpuRenderer(s, p) as r:
        r.render_spp(spp)
        rgb, sq, n = r.framebuffer()
    assert np.all(n == spp)
    mean = rgb / spp
    var = np.maximum(sq / spp - mean ** 2, 0) * spp / (spp - 1)
    z = _zscores(mean, np.sqrt(var / spp), f["mean"], f["stderr"])
    frac3 = float(np.mean(np.abs(z) > 3))
    print(f"{name}: mean z {z.mean():+.4f}, |z|>3 fraction {frac3:.4f}, max |z| {np.abs(z).max():.2f}", flush=True)
    # Gaussian tails give 0.27 % beyond 3 sigma; heavy-tailed path estimates allow up to 1.5 %.
    assert frac3 < 0.015
    # No systematic bias: the mean z-score over all pixel channels is ~N(0, 1/sqrt(n)).
    assert abs(z.mean()) < 5.0 / np.sqrt(z.size) + 0.02
    # Image-average radiance agrees within 4 standard errors of the difference (+0.1 % for FP32).
    npix = mean.shape[0] * mean.shape[1]
    img, img_ref = mean.mean(axis=(0, 1)), f["mean"].mean(axis=(0, 1))
    img_se = np.sqrt((var / spp).sum(axis=(0, 1)) + (f["stderr"] ** 2).sum(axis=(0, 1))) / npix
    print(f"{name}: image mean {img} oracle {img_ref} +- {img_se}", flush=True)
    assert np.all(np.abs(img - img_ref) < 4 * img_se + 1e-3 * np.abs(img_ref))


def test_cornell_parity_reference_mis(gpu_lib):
    render_parity("cornell64")


def test_cornell_parity_sorted_shade(gpu_lib, monkeypatch):
    """The shade kernel with its per-block sort by shader class renders the same image."""
    monkeypatch.setenv("TTGPU_SORT_SHADE", "1")
    render_parity("cornell32_consistent", mis=abi.MIS_CONSISTENT)
    render_parity("terrain32", builder=lambda w, h: configs.terrain_instances(w, h, cells=32, n_spheres=24, freq=3,
                                                                            sky=(256, 128)))


@pytest.mark.parametrize("shadow_in_trace,slot_order", [("0", "1"), ("1", "0"), ("0", "0")])
def test_traversal_modes_render_the_same_image(gpu_lib, monkeypatch, shadow_in_trace, slot_order):
    """Separate shadow launches and queues appended per block instead of selected in slot order give
    the default mode's image (shadow rays in the next closest-hit launch, slot-ordered queues) up to
    the order of the FP64 framebuffer sums: every path draws the same random numbers whichever kernel
    traces it, in whatever order."""
    def render():
        s = configs.terrain_instances(48, 32, cells=32, n_spheres=24, freq=3, sky=(256, 128))
        with GpuRenderer(s, abi.default_params(48, 32, spp=16, max_depth=8, seed=5)) as r:
            r.run()
            return r.mean_image()
    base = render()
    monkeypatch.setenv("TTGPU_SHADOW_IN_TRACE", shadow_in_trace)
    monkeypatch.setenv("TTGPU_SLOT_ORDER", slot_order)
    other = render()
    print(f"max |diff| {np.abs(other - base).max():.3e}, mean {base.mean():.4f}", flush=True)
    assert base.mean() > 0
    np.testing.assert_allclose(other, base, rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("algo", ["pt2_media", "pt"])
def test_queue_order_renders_the_same_image(gpu_lib, monkeypatch, algo):
    """Slot-ordered queues against per-block appends, in a participating medium (null-path
    tracking, shadow rays in their own launch) and with pt's light connections to the camera:
    the same image up to the order of the FP64 framebuffer sums."""
    def render():
        if algo == "pt":
            s = configs.cornell_box(32, 32)
            p = abi.default_params(32, 32, spp=16, max_depth=6, seed=7, algo=abi.ALGO_PT)
        else:
            s = configs.medium_sphere(32, 32)
            p = abi.default_params(32, 32, spp=16, max_depth=8, seed=7)
        with GpuRenderer(s, p) as r:
            r.run()
            return r.mean_image()
    base = render()
    monkeypatch.setenv("TTGPU_SLOT_ORDER", "0")
    monkeypatch.setenv("TTGPU_SORT_SHADE", "1")
    other = render()
    print(f"{algo}: max |diff| {np.abs(other - base).max():.3e}, mean {base.mean():.4f}", flush=True)
    assert base.mean() > 0
    np.testing.assert_allclose(other, base, rtol=1e-9, atol=1e-12)


def test_cornell_parity_consistent_mis(gpu_lib):
    render_parity("cornell32_consistent", mis=abi.MIS_CONSISTENT)


def test_cornell_parity_bsdf_only(gpu_lib):
    render_parity("cornell32_bsdf", mode=abi.SAMPLE_BSDF)


def test_terrain_env_map_parity(gpu_lib):
    # The benchmark scene at 32x32: HDR sky map with a sun disc (alias-table NEE on the GPU, CDF
    # inversion in the oracle), GGX / glass / mirror / Lambert on a heightfield and icospheres.
    render_parity("terrain32", builder=lambda w, h: configs.terrain_instances(w, h, cells=32, n_spheres=24, freq=3, sky=(256, 128)))


def test_run_schedule_and_image(gpu_lib):
    """Run(): doubling passes 1,2,4,... capped by max spp (SamplesPerPixelSchedule)."""
    s = configs.cornell_box(32, 24)
    p = abi.default_params(32, 24, spp=20)
    calls = []
    with GpuRenderer(s, p) as r:
        r.set_pass_callback(lambda complete: calls.append(complete))
        r.run()
        _, _, n = r.framebuffer()
        assert np.all(n == 20)  # 1 + 2 + 4 + 8 + 5
        assert calls == [True] * 5
        img = r.generate_image()
        assert img.shape == (24, 32, 3) and img.dtype == np.uint8 and img.max() > 0
        st = r.stats()
        assert st["total_spp"] == 20 and st["paths_traced"] == 32 * 24 * 20


def test_stop_before_run(gpu_lib):
    s = configs.cornell_box(16, 16)
    p = abi.default_params(16, 16, spp=64)
    with GpuRenderer(s, p) as r:
        r.request_stop()
        rc = r.run()
        assert rc == 4  # TTGPU_ERR_INTERRUPTED: no pass was started
        _, _, n = r.framebuffer()
        assert n.sum() == 0


def test_invalid_scene_rejected(gpu_lib):
    s = configs.cornell_box(8, 8)
    s.tri_material[0] = s.tri_material[0].copy()
    s.tri_material[0][0] = 99
    with pytest.raises(RuntimeError, match="material"):
        GpuRenderer(s, abi.default_params(8, 8))
