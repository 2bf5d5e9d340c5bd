"""Results are ordinary arrays with memory of their own: they stay what they
were while their owner renders on, however many are held, also after it is
closed, and a forked process has them too."""
import ctypes as C
import gc
import threading

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


def map_flags(array):
    """The flags of the memory mappings that hold the array's first and last byte."""
    flags, ends = [], (array.ctypes.data, array.ctypes.data + array.nbytes - 1)
    for line in open("/proc/self/smaps"):
        word = line.split(" ")[0]
        if "-" in word and ":" not in word:
            lo, hi = (int(x, 16) for x in word.split("-"))
            held = any(lo <= end < hi for end in ends)
        elif word == "VmFlags:" and held:
            flags += line.split()[1:]
    assert flags
    return flags


@pytest.mark.parametrize("width,height", [(64, 48), (640, 480), (1500, 700)])
def test_result_memory_is_the_callers(torch_cuda, width, height):
    r = renderer(width, height, spp=1)
    frame, _ = r.render_frame()
    r.render_samples(1, 1)
    again, _ = r.framebuffer()
    tile = r.render_task(wpt.Task(0, 0, 0, 1, 3, 5, width - 3, height - 5))
    host = wpt.HostScene("cornell-box")
    scene = wpt.Scene(host.desc(), device=True, owner=host)
    tasks = [wpt.batch_task(0, host.camera(width, height), width, height, x, 0, w, height, 0, 1, max_depth=4)
             for x, w in ((0, 1), (1, width // 2), (40, 24))]
    for a in [frame, again, tile] + wpt.Batch([scene]).render(tasks):
        assert a.base is None  # keeping one result keeps no other
        flags = map_flags(a)
        assert "dc" not in flags and "sh" not in flags, flags  # copied on fork


@pytest.mark.parametrize("width,height", [(418, 418), (419, 418), (836, 418), (1277, 719)])
def test_whole_frames_from_several_threads(torch_cuda, width, height):
    """Frames just below and above the size read in pieces, of one piece and
    of several with a remainder, into ordinary memory, at odd addresses too,
    and into page-locked memory."""
    r = renderer(width, height, spp=1)
    r.render_samples(0, 1)
    want = r.render_task(wpt.Task(0, 0, 0, 1, 0, 0, width, height))
    got = [None] * 4

    def read(k):
        got[k] = r.framebuffer()[0]

    threads = [threading.Thread(target=read, args=(k,)) for k in range(len(got))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    lib, block = wpt.library(), C.c_void_p()
    wpt.check(lib.wpt_host_alloc(want.nbytes, C.byref(block)), "wpt_host_alloc")
    wpt.check(lib.wpt_renderer_read_framebuffer(r._h, block, None), "wpt_renderer_read_framebuffer")
    locked = np.ctypeslib.as_array(C.cast(block, C.POINTER(C.c_float)), want.shape).copy()
    wpt.check(lib.wpt_host_free(block), "wpt_host_free")
    assert all(np.array_equal(g, want) for g in got + [locked])
    for shift in (1, 2, 3):
        odd = np.full(want.size + 8, -1.0, np.float32)
        wpt.check(lib.wpt_renderer_read_framebuffer(r._h, odd[shift:].ctypes.data, None), "wpt_renderer_read_framebuffer")
        assert np.array_equal(odd[shift:shift + want.size], want.ravel())
        assert np.all(odd[:shift] == -1.0) and np.all(odd[shift + want.size:] == -1.0)
