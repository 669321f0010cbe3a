"""The two-launch slot selection (chunk counts scanned by the last block, queue and regeneration in
one scatter) against the appended queues, at wavefront sizes around its chunk (1024 slots, 16 flags
per lane) and block (16 chunks) edges, above 2^20 slots, where each thread of the last block scans
several chunks (two and three here), and with passes that refill the slots."""
import numpy as np
import pytest

from naivetrace_amd import abi, configs
from naivetrace_amd.renderer import GpuRenderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wavefront", [1, 15, 16, 17, 1023, 1024, 1025, 16383, 16384, 16385, 33001, (1 << 20) + 1,
                                       (1 << 21) + 1025])
def test_slot_selection_renders_the_appended_queues_image(gpu_lib, monkeypatch, wavefront):
    w, h = (5, 3) if wavefront < 1000 else (97, 61) if wavefront < 1 << 20 else (640, 512)
    spp = 3 if wavefront < 1000 else 8

    def render():
        p = abi.default_params(w, h, max_depth=6, seed=11)
        p.wavefront_paths = wavefront
        with GpuRenderer(configs.cornell_box(w, h), p) as r:
            r.render_spp(spp)
            r.render_spp(1)
            rgb, _, n = r.framebuffer()
            st = r.stats()
            return rgb, n, (st["rays_closest"], st["rays_shadow"], st["paths_traced"])
    rgb, n, rays = render()
    monkeypatch.setenv("TTGPU_SLOT_ORDER", "0")
    rgb0, n0, rays0 = render()
    assert np.all(n == spp + 1) and np.array_equal(n, n0)
    assert rays == rays0
    assert rgb.sum() > 0
    # The same paths: only the order of the FP64 sums differs (at most 9 terms per pixel).
    np.testing.assert_allclose(rgb, rgb0, rtol=1e-12, atol=1e-15)
