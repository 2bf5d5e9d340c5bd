"""Results read back into page-locked blocks: arrays stay what they were while
their owner renders on, however many are held, also after it is closed."""
import gc

import numpy as np
import pytest

import wpt

pytestmark = pytest.mark.gpu


def renderer(width=640, height=480, spp=4, **kw):
    host = wpt.HostScene("cornell-box")
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    cfg = wpt.render_config(width, height, spp=spp, max_depth=4, rr_start=3, **kw)
    return wpt.Renderer(scene, host.camera(width, height), cfg)


@pytest.mark.parametrize("held", [1, 2, 3, 7])
def test_held_frames_keep_their_values(torch_cuda, held):
    r = renderer(64, 48)
    frames, copies = [], []
    for k in range(2 * held):
        r.reset()
        r.render_samples(k, 1)
        image, n = r.framebuffer()
        assert n == k + 1 and image.flags.writeable and image.shape == (48, 64, 3)
        frames.append(image)
        copies.append(image.copy())
        if len(frames) > held:
            frames.pop(0), copies.pop(0)
            gc.collect()
        for a, b in zip(frames, copies):
            assert np.array_equal(a, b)
    views = [f[3:9, 5:7] for f in frames]
    expect = [c[3:9, 5:7] for c in copies]
    del frames, image
    r.close()
    gc.collect()
    for a, b in zip(views, expect):
        assert np.array_equal(a, b)
    assert not np.array_equal(views[0], views[-1]) or held == 1


def test_batch_results_are_separate(torch_cuda):
    host = wpt.HostScene("cornell-box")
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    cam = host.camera(128, 96)
    batch = wpt.Batch([scene])
    tasks = [wpt.batch_task(0, cam, 128, 96, x, 5, 31, 17, 0, 2, max_depth=4) for x in (0, 40, 90)]
    first = batch.render(tasks)
    keep = [o.copy() for o in first]
    second = batch.render(tasks[::-1])
    first[1][:] = -1.0
    assert np.array_equal(first[0], keep[0]) and np.array_equal(first[2], keep[2])
    assert all(np.array_equal(a, b) for a, b in zip(second, keep[::-1]))
    assert batch.render([]) == []
