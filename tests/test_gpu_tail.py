"""The staged scheduler's two ways through a pass: queues of more than 131,072
paths bounce by bounce, smaller ones by the kernel that takes each path to its
end.  Frames just below, at and above the limit, one of whose later bounces
crosses it, equal the oracle's bit for bit, with its query counts; a batch of
tasks on either side equals the frames' tiles."""
import numpy as np
import pytest

import test_gpu_terrain as terrain
import wpt

pytestmark = pytest.mark.gpu

LIMIT = 131072
SIZES = [(512, LIMIT // 512, 1), (513, LIMIT // 512, 1), (509, 103, 5)]


def check(oracle_mod, scene, cam, cfg):
    r = wpt.Renderer(scene, cam, cfg)
    image, _ = r.render_frame()
    st = r.stats()
    again, _ = r.render_frame()
    r.close()
    want, ost = oracle_mod.Oracle(scene).render(cam, cfg)
    assert np.array_equal(image, want), np.abs(image - want).max()
    assert np.array_equal(again, want)
    assert (st.closest_queries, st.shadow_queries) == (ost.closest_queries, ost.shadow_queries)
    return st


@pytest.mark.parametrize("width,height,spp", SIZES)
@pytest.mark.parametrize("preset,freq", [("cornell-box", 0), ("sphere-field", 12), ("prism", 0)])
def test_frames_around_the_limit(torch_cuda, oracle_mod, preset, freq, width, height, spp):
    host = wpt.HostScene(preset, icosphere_frequency=freq)
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    cam = host.camera(width, height)
    cfg = wpt.render_config(width, height, spp=spp, max_depth=9, rr_start=3)
    st = check(oracle_mod, scene, cam, cfg)
    assert st.queue_counts[0] == width * height * spp
    cfg.mode = wpt.MODE_PERSISTENT
    r = wpt.Renderer(scene, cam, cfg)
    r.render_frame()
    assert list(r.stats().queue_counts) == list(st.queue_counts)


@pytest.mark.parametrize("width,height,spp", SIZES)
def test_radiance_events_around_the_limit(torch_cuda, oracle_mod, tmp_path, width, height, spp):
    host = wpt.HostScene(terrain.small_manifest(tmp_path))
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    rc, _ = terrain.config(terrain.small_manifest(tmp_path), width, height, spp, 20000)
    check(oracle_mod, scene, host.camera(width, height), rc)


def test_batch_passes_on_both_sides(torch_cuda):
    host = wpt.HostScene("sphere-field", icosphere_frequency=12)
    cornell = wpt.HostScene("cornell-box")
    scenes = [wpt.Scene(h.desc(), device=True, owner=h) for h in (host, cornell)]
    cams = [h.camera(640, 480) for h in (host, cornell)]
    shapes = [(0, 300, 220, 3), (1, 31, 17, 2), (0, 640, 480, 1), (1, 257, 129, 5)]
    tasks = [wpt.batch_task(s, cams[s], 640, 480, 0, 0, w, h, 2, n, max_depth=8, rr_start=3) for s, w, h, n in shapes]
    outs = wpt.Batch(scenes, scheduler=wpt.BATCH_STAGED).render(tasks)
    for (s, w, h, n), out in zip(shapes, outs):
        cfg = wpt.render_config(640, 480, spp=n, max_depth=8, rr_start=3, mode=wpt.MODE_REGENERATE)
        r = wpt.Renderer(scenes[s], cams[s], cfg)
        r.reset()
        r.render_samples(2, n)
        image, _ = r.framebuffer()
        assert np.array_equal(out, image[:h, :w])


def renderer(width=640, height=480, spp=4, **kw):
    host = wpt.HostScene("cornell-box")
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    cfg = wpt.render_config(width, height, spp=spp, max_depth=4, rr_start=3, **kw)
    return wpt.Renderer(scene, host.camera(width, height), cfg)


@pytest.mark.parametrize("width,height,samples", [(1, 1, 1), (31, 17, 2), (512, 256, 1), (512, 257, 1), (640, 480, 3)])
def test_small_passes_of_a_large_renderer(torch_cuda, width, height, samples):
    r = renderer()
    tile = r.render_task(wpt.Task(0, 0, 1, samples, 640 - width, 480 - height, width, height))
    r.reset()
    r.render_samples(1, samples)
    image, n = r.framebuffer()
    assert n == 1 + samples
    assert np.array_equal(tile, image[480 - height:, 640 - width:])
    tiled = renderer(tile=(200, 130))
    tiled.render_samples(1, samples)
    again, n = tiled.framebuffer()
    assert n == 1 + samples and np.array_equal(again, image)
