"""GPU tests of shading in material order where paths meet an environment map or the radiance cache: the same
image, and the same cache records, as in queue order."""
import numpy as np
import pytest

import scenes
import vt

pytestmark = pytest.mark.gpu


def _scene(ctx, env):
    mesh, mats = scenes.materials_cornell("opaque")
    scene = ctx.set_mesh(mesh)
    scene.set_materials(scenes.vt_materials(mats))
    if env:
        scene.set_environment(scenes.sky_map())
    return scene


@pytest.mark.parametrize("w,h", [(33, 31), (73, 61)])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_environment(gpu_ctx, w, h, mode):
    scene = _scene(gpu_ctx, True)
    images = []
    for sort in (False, True):
        r = vt.Renderer(gpu_ctx)
        r.render(scene, w, h, vt.orbit_eye(), (0.0, -0.1, 0.0), 42.0, max_depth=4, samples=2, sample_index=1,
                 sampling_mode=mode, env_strength=1.0, material_sort=sort)
        images.append(r.readback())
        r.close()
    scene.close()
    print(f"environment {w}x{h} mode {mode}: mean {images[0][..., :3].mean():.5f}", flush=True)
    assert images[0][..., :3].mean() > 0.01
    assert np.array_equal(images[0], images[1])


@pytest.mark.parametrize("w,h", [(33, 31), (97, 61)])
@pytest.mark.parametrize("mode", [0, 1])
def test_cache_records(gpu_ctx, w, h, mode):
    # A frozen cache, so that the order of the records cannot reach the image.
    scene = _scene(gpu_ctx, False)
    cache = vt.NRC(gpu_ctx, seed=3)
    images, records = [], []
    for sort in (False, True):
        r = vt.Renderer(gpu_ctx)
        r.set_cache(cache)
        r.render(scene, w, h, vt.orbit_eye(), (0.0, -0.1, 0.0), 42.0, max_depth=5, samples=1, sample_index=2,
                 sampling_mode=mode, cache=2, train_period=2, material_sort=sort)
        images.append(r.readback())
        x, t, made = r.cache_records()
        assert made == len(x)
        rows = np.concatenate([x, t], axis=1).view(np.uint32)
        records.append(rows[np.lexsort(rows.T)])
        r.close()
    scene.close()
    cache.close()
    print(f"cache {w}x{h} mode {mode}: {len(records[0])} records", flush=True)
    assert len(records[0]) > 20
    assert np.array_equal(images[0], images[1])
    assert np.array_equal(records[0], records[1])
