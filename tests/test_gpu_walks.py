"""GPU tests of the interleaved ray walks of the staged scheduler at the sizes
where a wave's refill can go wrong: frames whose paths are one ray, just
below, at and above a wave and a workgroup, and a few rays beyond the resident
grid's first round.  The oracle's image is the expectation, bit for bit (a
path's arithmetic does not depend on its wave), and its query counts."""
import numpy as np
import pytest

import wpt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset,freq", [("sphere-field", 12), ("prism", 0)])
@pytest.mark.parametrize("width,height,spp,block", [(1, 1, 1, 64), (63, 1, 1, 64), (8, 8, 1, 64), (65, 1, 1, 256),
                                                    (257, 1, 1, 256), (17, 13, 7, 512)])
def test_frames_around_wave_sizes(torch_cuda, oracle_mod, preset, freq, width, height, spp, block):
    host = wpt.HostScene(preset, icosphere_frequency=freq)
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    cam = host.camera(width, height)
    cfg = wpt.render_config(width, height, spp=spp, max_depth=12, rr_start=3, block_size=block)
    r = wpt.Renderer(scene, cam, cfg)
    image, samples = r.render_frame()
    want, stats = oracle_mod.Oracle(scene).render(cam, cfg)
    got = r.stats()
    assert samples == spp
    assert np.array_equal(image, want), np.abs(image - want).max()
    assert (got.closest_queries, got.shadow_queries) == (stats.closest_queries, stats.shadow_queries)
