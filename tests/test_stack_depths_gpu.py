"""GPU tests of every traversal stack the launchers tell apart: hierarchies whose depth asks for it (asserted),
traced one-level and instanced against the oracle's brute force bit for bit, and rendered single and batched
against the flat binary hierarchy, which has none of these stacks."""
import numpy as np
import pytest

import oracle
from oracle import instances as oinst
import scenes
import vt

pytestmark = pytest.mark.gpu

# Triangles of a series, and the pending groups (depth - 1) its hierarchy may need: the stacks of 8, 10, 12, 16
# and 24 groups.
STACKS = [(60, 1, 8), (90, 9, 10), (100, 11, 12), (115, 13, 16), (150, 17, 24)]


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda:0")


def _same(got, ref, what, keys=("t", "b1", "b2", "face")):
    for k in keys:
        g = got[k].cpu().numpy()
        assert (g == ref[k].astype(g.dtype, copy=False)).all(), f"{what}: {k}"


@pytest.mark.parametrize("count,low,high", STACKS)
def test_traces(gpu_ctx, count, low, high):
    tri = scenes.series(count)
    v, f = scenes.mesh_from_triangles(tri.astype(np.float32))
    scene = gpu_ctx.set_mesh(vt.Mesh(v, f))
    assert low <= scene.info["depth"] - 1 <= high
    rays = scenes.series_rays(tri, 8000, count)
    ref = oracle.Scene(v, f, with_bvh=False).closest(rays, mode=1)
    hit = ref["face"] >= 0
    print(f"{count} triangles, depth {scene.info['depth']}, {int(hit.sum())} hits", flush=True)
    assert hit.sum() > 500
    _same(scene.trace_closest(_dev(rays)), ref, "closest")
    assert np.array_equal(scene.trace_any(_dev(rays)).cpu().numpy() != 0, hit)
    gpu_ctx.check()
    scene.close()


@pytest.mark.parametrize("count,low,high", STACKS)
def test_renders(gpu_ctx, count, low, high):
    light = np.array([[[-2, 3, -2], [4, 3, -2], [-2, 3, 4]]])
    v, f = scenes.mesh_from_triangles(np.concatenate([scenes.series(count), light]).astype(np.float32))
    f[-1, 3] = 1
    mats = [vt.material(0, (0.7, 0.6, 0.5)), vt.material(3, (0, 0, 0), (5.0, 5.0, 5.0))]
    view = (64, 48, (0.9, 1.1, -1.2), (0.2, 0.2, 0.0), 60.0)
    images, built = [], []
    for collapse in (2, 0):
        scene = gpu_ctx.set_mesh(vt.Mesh(v, f), collapse=collapse)
        scene.set_materials(mats)
        r = vt.Renderer(gpu_ctx)
        r.render(scene, *view, max_depth=5, samples=2, sample_index=1)
        images.append(r.readback())
        r.close()
        built.append(scene)
    assert low <= built[1].info["depth"] - 1 <= high
    print(f"{count} triangles, depth {built[1].info['depth']}, mean {images[0][..., :3].mean():.5f}", flush=True)
    assert images[0][..., :3].mean() > 0.001
    assert np.array_equal(images[0], images[1])
    # As the batch tests compare a job with its single image: the same samples, float order apart.
    b = vt.Batch(gpu_ctx, [(built[1], *view)], max_depth=5)
    b.render(2)
    assert np.isclose(b.readback(0), images[1], rtol=1e-4, atol=1e-6).all(axis=2).mean() > 0.999
    gpu_ctx.check()
    b.close()
    for s in built:
        s.close()


# Instances and triangles, and the groups both levels need together: the stacks of 10, 16, 24 and 40 groups.
@pytest.mark.parametrize("count,instances,low,high", [(30, 8, 1, 10), (60, 60, 11, 16), (100, 100, 17, 24), (150, 300, 25, 40)])
def test_instances(gpu_ctx, count, instances, low, high):
    tri = scenes.series(count)
    v, f = scenes.mesh_from_triangles(tri.astype(np.float32))
    built = gpu_ctx.set_mesh(vt.Mesh(v, f))
    inst = []
    for a in 0.8 ** np.arange(instances):
        w = np.zeros((3, 4), np.float32)
        w[:, :3] = np.eye(3) * max(0.3 * a, 1e-5)
        w[:, 3] = (2 * a - 1, -a, 0.5 * a)
        inst.append((0, w))
    tl = vt.Tlas(gpu_ctx, [(built, w) for _, w in inst])
    info = tl.info
    groups = max(info["depth"] - 1, 1) + max(info["blas_depth"] - 1, 1)
    print(f"{count} triangles, {instances} instances: depths {info['depth']} and {info['blas_depth']}", flush=True)
    assert low <= groups <= high
    # Rays at the series of the larger instances, in the world.
    local = scenes.series_rays(tri, 6000, instances)
    pick = np.stack([w for _, w in inst])[np.random.default_rng(1).integers(0, min(instances, 20), 6000)].astype(np.float64)
    rays = local.copy()
    rays[0:3] = (np.einsum("nij,jn->in", pick[:, :, :3], local[0:3].astype(np.float64)) + pick[:, :, 3].T).astype(np.float32)
    ref = oinst.closest([oracle.Scene(v, f, with_bvh=False)], inst, rays)
    hit = ref["face"] >= 0
    assert hit.sum() > 500
    got = tl.trace_closest(_dev(rays))
    _same(got, ref, "closest")
    assert np.array_equal(got["instance"].cpu().numpy().view(np.uint32), ref["instance"].astype(np.uint32))
    assert np.array_equal(tl.trace_any(_dev(rays)).cpu().numpy() != 0, hit)
    gpu_ctx.check()
    tl.close()
    built.close()
