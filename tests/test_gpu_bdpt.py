"""Bidirectional path tracing (TTGPU_ALGO_BDPT) on the GPU, through the C ABI.

* Parity with the oracle's renders (tests/golden/*_bdpt_oracle.npz): the Cornell box (consistent
  Russian roulette) and a wide view with a point light and a dome (the reference's roulette
  placement and pixel lookup); standard errors from independent batches on both sides.
* Closed forms: furnace L_e (1 - rho^d) / (1 - rho), the furnace with a glass and a lossless
  mirror sphere, an emitter filling the view, a plane under a dome.
* The reference's Russian-roulette placement biases the furnace upwards beyond depth 5 exactly as
  in the oracle; scenes the kernel does not support are rejected.
"""
import os

import numpy as np
import pytest

from naivetrace_amd import abi, configs
from naivetrace_amd.renderer import GpuRenderer, TTGpuError
from naivetrace_amd.scene import Scene, flat, spectrum_to_rgb
from test_bdpt import specular_furnace
from test_gpu_parity import GOLDEN, _zscores
from test_gpu_pt import gpu_batches
from test_oracle import fog_furnace_scene, furnace_scene
from test_pt import emitter_wall_scene
from golden.make_oracle_images import BDPT_FIXTURES

pytestmark = pytest.mark.gpu


def _params(w, h, depth, mis=abi.MIS_CONSISTENT, seed=11):
    p = abi.default_params(w, h, max_depth=depth, seed=seed, algo=abi.ALGO_BDPT)
    p.mis_mode = mis
    return p


def _image(mean, se, w, h):
    return mean.mean(axis=(0, 1)), np.sqrt((se ** 2).sum(axis=(0, 1))) / (w * h)


@pytest.mark.parametrize("name", list(BDPT_FIXTURES))
def test_gpu_bdpt_parity(gpu_lib, name):
    build, w, h, batches, spp, depth, mis, mode = BDPT_FIXTURES[name]
    f = np.load(os.path.join(GOLDEN, f"{name}_oracle.npz"))
    assert int(f["mis_mode"]) == mis and int(f["algo"]) == abi.ALGO_BDPT
    print(f"bdpt parity {name}: {batches} x {spp} spp", flush=True)
    mean, se = gpu_batches(build(w, h), _params(w, h, depth, mis), batches, spp)
    z = _zscores(mean, se, f["mean"], f["stderr"])
    frac3 = float(np.mean(np.abs(z) > 3))
    print(f"{name}: mean z {z.mean():+.4f}, |z|>3 fraction {frac3:.4f}, max |z| {np.abs(z).max():.2f}", flush=True)
    assert frac3 < 0.04
    assert abs(z.mean()) < 5.0 / np.sqrt(z.size) + 0.03
    img, img_se = _image(mean, se, w, h)
    ref, ref_se = _image(f["mean"], f["stderr"], w, h)
    print(f"{name}: image mean {img} oracle {ref} +- {np.sqrt(img_se ** 2 + ref_se ** 2)}", flush=True)
    assert np.all(np.abs(img - ref) < 4 * np.sqrt(img_se ** 2 + ref_se ** 2) + 1e-3 * np.abs(ref))


@pytest.mark.parametrize("depth", [3, 8, 16])
def test_gpu_bdpt_furnace_closed_form(gpu_lib, depth):
    rho = 0.5
    img, img_se = _image(*gpu_batches(furnace_scene(rho), _params(8, 8, depth), 8, 128), 8, 8)
    expected = spectrum_to_rgb(flat(sum(rho ** k for k in range(depth))))
    print(f"bdpt furnace depth {depth}: {img} +- {img_se} expected {expected}", flush=True)
    assert np.all(np.abs(img - expected) < 4 * img_se + 2e-3 * expected)


def test_gpu_bdpt_specular_furnace(gpu_lib):
    rho = 0.5
    img, img_se = _image(*gpu_batches(specular_furnace(rho), _params(8, 8, 16), 8, 256), 8, 8)
    expected = spectrum_to_rgb(flat(sum(rho ** k for k in range(16))))
    print(f"bdpt specular furnace: {img} +- {img_se} expected {expected}", flush=True)
    assert np.all(np.abs(img - expected) < 4 * img_se + 3e-3 * expected)


def test_gpu_bdpt_reference_russian_roulette_bias(gpu_lib):
    s = furnace_scene(0.5)
    ref, ref_se = _image(*gpu_batches(s, _params(8, 8, 8, abi.MIS_REFERENCE), 8, 256), 8, 8)
    con, con_se = _image(*gpu_batches(s, _params(8, 8, 8, abi.MIS_CONSISTENT, seed=12), 8, 256), 8, 8)
    diff = (ref - con) / np.sqrt(ref_se ** 2 + con_se ** 2)
    print(f"bdpt roulette placement: reference {ref} consistent {con} z {diff}", flush=True)
    assert np.all(diff > 6)


def test_gpu_bdpt_visible_emitter_and_dome(gpu_lib):
    L = 2.0
    mean, se = gpu_batches(emitter_wall_scene(L), _params(8, 6, 4), 8, 256)
    expected = spectrum_to_rgb(flat(L))
    assert np.all(np.abs(mean - expected) < 5 * se + 2e-3 * expected)
    s = Scene()
    rho, Ld = 0.6, 1.5
    m = s.add_material(shader=s.add_shader(abi.SHADER_DIFFUSE, reflectance=flat(rho)))
    big = 1e4
    s.add_quad([-big, 0, big], [big, 0, big], [big, 0, -big], [-big, 0, -big], m)
    s.add_dome([0, 1, 0], flat(Ld))
    s.set_camera([0, 1, 0], [0, 0, -0.2], [0, 0, -1], 30.0)
    img, img_se = _image(*gpu_batches(s, _params(4, 4, 3), 8, 512), 4, 4)
    expected = spectrum_to_rgb(flat(rho * Ld))
    assert np.all(np.abs(img - expected) < 4 * img_se + 2e-3)


def test_gpu_bdpt_rejects_unsupported(gpu_lib):
    with pytest.raises(TTGpuError, match="surface scenes"):
        GpuRenderer(fog_furnace_scene(0.5), _params(4, 4, 8))
    with pytest.raises(TTGpuError, match="max_ray_depth"):
        GpuRenderer(furnace_scene(0.5), _params(4, 4, 17))
    s = configs.cornell_box(8, 8)
    s.set_camera([0.0, 1.0, 3.4], [0.0, 1.0, 0.0], [0.0, 1.0, 0.0], 40.0, kind=abi.CAMERA_FISHEYE)
    with pytest.raises(TTGpuError, match="pinhole"):
        GpuRenderer(s, _params(8, 8, 8))


@pytest.mark.parametrize("w,h,spp,depth", [(1, 1, 3, 2), (13, 7, 5, 16), (91, 90, 4, 3), (128, 64, 4, 3), (257, 511, 3, 16),
                                              (641, 421, 4, 3)])
def test_gpu_bdpt_chunks_and_wave_edges(gpu_lib, w, h, spp, depth):
    """One pass (the last two span two chunks, of 2^18 and 2^20 samples, and end inside a wave) equals
    the sum of 1-spp passes: each sample draws the same numbers wherever it lies in a chunk.  Frames of
    8190 pixels take their samples by atomics, of 8192 and more by a thread per pixel.  A sample's sum
    runs over at most 136 connections in another order, in FP64, and is rounded to FP32 once."""
    scene = configs.cornell_box(w, h)

    def render(passes):
        with GpuRenderer(scene, _params(w, h, depth)) as r:
            for n in passes:
                r.render_spp(n)
            rgb, sq, n = r.framebuffer()
            return rgb, sq, n, r.stats()["paths_traced"]
    a, a2, na, pa = render([spp])
    b, b2, nb, pb = render([1] * spp)
    assert np.all(na == spp) and np.array_equal(na, nb) and pa == pb == w * h * spp
    if w > 100:
        assert a.sum() > 0
    np.testing.assert_allclose(a, b, rtol=spp * 2.0 ** -23, atol=1e-12)
    np.testing.assert_allclose(a2, b2, rtol=spp * 2.0 ** -22, atol=1e-12)


def _sample_bytes(depth):
    """Workspace of a sample: three vertices of 96 B per path vertex, its connections, its sums."""
    return 3 * 96 * (depth + 1) + 4 * depth * (depth + 1) // 2 + 32


@pytest.mark.parametrize("depth,wavefront,expected", [
    (16, 0, 1 << 18), (8, 0, (_sample_bytes(16) << 18) // _sample_bytes(8)), (2, 0, 1 << 20), (2, 1 << 21, 1 << 20),
    (8, 20001, 20001), (8, 1, 1 << 13)])
def test_gpu_bdpt_wavefront_paths_bound_the_workspace(gpu_lib, depth, wavefront, expected):
    """The samples in flight: what 2^18 take at depth 16, up to 2^20, or the caller's wavefront size,
    which bounds a handle's memory; the image does not depend on it.  A sample's FP64 sum is rounded to
    FP32 once, in whatever order its connections arrive."""
    w, h, spp = 97, 65, 5

    def render(paths):
        p = _params(w, h, depth)
        p.wavefront_paths = paths
        with GpuRenderer(configs.cornell_box(w, h), p) as r:
            r.render_spp(spp)
            rgb, _, n = r.framebuffer()
            assert np.all(n == spp)
            return rgb, r.stats()
    rgb, st = render(wavefront)
    assert st["wavefront_paths"] == expected
    assert st["state_bytes"] < expected * _sample_bytes(depth) + 4096
    ref, _ = render(0)
    np.testing.assert_allclose(rgb, ref, rtol=spp * 2.0 ** -23, atol=1e-12)
