"""GPU tests of image readback: sizes around the step from one copy to a staged one and around its chunks,
destinations at odd addresses, in pinned memory and larger than the image, and several threads reading images
of one context at once -- every way gives the bytes that a direct copy to pinned memory gives."""
import ctypes
import threading

import numpy as np
import pytest

import vt

pytestmark = pytest.mark.gpu


def _image(ctx, scene, w, h):
    r = vt.Renderer(ctx)
    r.render(scene, w, h, vt.orbit_eye(), (0.0, -0.1, 0.0), 42.0, max_depth=2, samples=1, sample_index=1)
    return r


def _scene(ctx):
    scene = ctx.set_mesh(vt.cornell())
    scene.set_materials(vt.cornell_materials(17.0))
    return scene


def _read(r, address, nbytes):
    assert vt.load().vt_accum_readback(r._h, ctypes.c_void_p(address), nbytes) == 0


def _pinned(r, count):
    import torch
    t = torch.empty(count, dtype=torch.float32, pin_memory=True)
    _read(r, t.data_ptr(), 4 * count)
    return t.numpy()


# 16 bytes a pixel: staged from 8 MiB (524288 pixels) on, in chunks of 512 KiB, from 16 MiB on of 1 MiB.
@pytest.mark.parametrize("w,h", [(1, 1), (512, 512), (524287, 1), (1024, 512), (524289, 1), (1024, 640), (1024, 1024), (1031, 1021)])
def test_sizes_and_destinations(gpu_ctx, w, h):
    scene = _scene(gpu_ctx)
    r = _image(gpu_ctx, scene, w, h)
    n = 4 * w * h
    ref = _pinned(r, n)
    assert (ref.reshape(h, w, 4)[..., 3] == ref[3]).all()
    for k in range(2):
        assert np.array_equal(r.readback().reshape(-1).view(np.uint32), ref.view(np.uint32)), k
    # At an address of 1 mod 4, in a buffer with room on both sides, which stays as it was.
    raw = np.full(4 * n + 64, 0xA5, np.uint8)
    _read(r, raw.ctypes.data + 33, raw.nbytes - 33)
    assert np.array_equal(raw[33:33 + 4 * n].view(np.uint8), ref.view(np.uint8))
    assert (raw[:33] == 0xA5).all() and (raw[33 + 4 * n:] == 0xA5).all()
    r.close()
    scene.close()


def test_threads(gpu_ctx):
    scene = _scene(gpu_ctx)
    renderers = [_image(gpu_ctx, scene, 800 + 60 * k, 700) for k in range(4)]
    refs = [_pinned(r, 4 * r.size[0] * r.size[1]) for r in renderers]
    bad = []

    def work(k):
        for _ in range(6):
            if not np.array_equal(renderers[k].readback().reshape(-1), refs[k], equal_nan=True):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for r in renderers:
        r.close()
    scene.close()
