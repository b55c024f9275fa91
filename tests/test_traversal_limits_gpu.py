"""GPU tests of the traversal at the limits of the float range, on every route that reaches it: closest and
any hit, the counting kernels, instanced meshes, single-image and batched rendering."""
import numpy as np
import pytest

import oracle
from oracle import instances as oinst
import scenes
import vt

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda:0")


def _same(got, ref, what):
    for k in ("t", "b1", "b2", "face"):
        g, r = got[k].cpu().numpy(), ref[k]
        assert ((g == r) | (np.isnan(g) & np.isnan(r))).all(), f"{what}: {k}"


def _check(ctx, v, f, rays, what):
    import torch
    scene = ctx.set_mesh(vt.Mesh(v, f))
    ref = oracle.Scene(v, f, with_bvh=False).closest(rays, mode=1)
    hit = ref["face"] >= 0
    print(f"{what}: {len(f)} triangles, {rays.shape[1]} rays, {int(hit.sum())} hits", flush=True)
    d = _dev(rays)
    _same(scene.trace_closest(d), ref, what)
    assert np.array_equal(scene.trace_any(d).cpu().numpy() != 0, hit), what
    counters = torch.zeros(2, dtype=torch.int64, device="cuda:0")
    _same(scene.trace_stats_noalloc(d, counters), ref, what)
    assert np.array_equal(scene.trace_stats_noalloc(d, counters, any_hit=True).cpu().numpy() != 0, hit), what
    ctx.check()
    scene.close()


# Either side of the size from which node boxes are scaled (2^82 = 4.8e24), where a grid step times 2^24 and
# 1e8 would overflow (5e25), and where the step itself would.
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("length", [4.7e24, 4.9e24, 1e26, 1e28, 1e32, 1e37])
def test_long_strips(gpu_ctx, length, axis):
    v, f, rays = scenes.long_strip(length, axis)
    _check(gpu_ctx, v, f, rays, f"strip {length:g} along {axis}")


@pytest.mark.parametrize("length,scale", [(1e22, 1e-16), (1e28, 1e-22)])
def test_long_strip_instanced(gpu_ctx, length, scale):
    # The strip brought back to 1e6 by its instances' transforms, beside an ordinary mesh.
    import torch
    strip = scenes.long_strip(length, 2)
    other = scenes.scattered_triangles(60, seed=4)
    world = np.zeros((3, 4), np.float32)
    world[0, 0], world[1, 1], world[2, 2] = 1000.0, 1000.0, scale
    moved, plain = world.copy(), np.eye(3, 4, dtype=np.float32)
    moved[1, 3] = -2000.0
    inst = [(0, world), (1, plain), (0, moved)]
    rays = strip[2].copy()
    rays[0:2] *= 1000.0
    rays[2] *= scale
    rays = np.concatenate([rays, scenes.random_rays(2000, 5)], axis=1)
    meshes = [strip[:2], other]
    built = [gpu_ctx.set_mesh(vt.Mesh(v, f)) for v, f in meshes]
    tl = vt.Tlas(gpu_ctx, [(built[a], w) for a, w in inst])
    ref = oinst.closest([oracle.Scene(v, f, with_bvh=False) for v, f in meshes], inst, rays)
    hit = ref["face"] >= 0
    print(f"instanced strip {length:g}: {int(hit.sum())} hits, {int(hit[:64].sum())} on the strip", flush=True)
    assert hit[:64].all()
    _same(tl.trace_closest(_dev(rays)), ref, "closest")
    assert np.array_equal(tl.trace_any(_dev(rays)).cpu().numpy() != 0, hit)
    torch.cuda.synchronize()
    gpu_ctx.check()
    tl.close()
    for s in built:
        s.close()


def test_render_with_far_geometry(gpu_ctx):
    # One triangle 1e27 away along x makes the boxes of the whole scene scaled.  The flat binary hierarchy has no such
    # boxes, and the same hits make the same image; a batch renders it too, as a single image to the batch
    # tests' bounds.
    mesh = vt.cornell()
    v = np.concatenate([mesh.vertices, np.zeros((3, 8), np.float32)])
    n = len(mesh.vertices)
    v[n:, :3] = np.array([[1e27, -0.5, 0.0], [1.1e27, -0.5, 0.0], [1e27, 0.5, 0.0]])
    v[n:, 4] = 1.0
    f = np.concatenate([mesh.faces, np.array([[n, n + 1, n + 2, 0]], np.uint32)])
    view = (48, 40, vt.orbit_eye(), (0.0, -0.1, 0.0), 42.0)
    images, built = [], []
    for collapse in (2, 0):
        scene = gpu_ctx.set_mesh(vt.Mesh(v, f), collapse=collapse)
        scene.set_materials(vt.cornell_materials(17.0))
        r = vt.Renderer(gpu_ctx)
        r.render(scene, *view, max_depth=5, samples=2, sample_index=1)
        images.append(r.readback())
        r.close()
        built.append(scene)
    print(f"mean {images[0][..., :3].mean():.6f}", flush=True)
    assert images[0][..., :3].mean() > 0.01
    assert np.array_equal(images[0], images[1])
    b = vt.Batch(gpu_ctx, [(built[1], *view)], max_depth=5)
    b.render(2)
    assert np.isclose(b.readback(0), images[0], rtol=1e-4, atol=1e-6).all(axis=2).mean() > 0.999
    b.close()
    for s in built:
        s.close()


@pytest.mark.parametrize("distance", [2.8e36, 3e36, 3.4e38])
def test_far_origins(gpu_ctx, distance):
    # They enter nothing (the node count shows it); the rays among them that do hit keep doing so.
    v, f = scenes.scattered_triangles(500, seed=2)
    far = scenes.far_rays(distance)
    scene = gpu_ctx.set_mesh(vt.Mesh(v, f))
    assert scene.trace_stats(_dev(far)) == (far.shape[1], 0)
    assert scene.trace_stats(_dev(far), any_hit=True) == (far.shape[1], 0)
    scene.close()
    _check(gpu_ctx, v, f, np.concatenate([far, scenes.random_rays(1000, 2)], axis=1), f"origins at {distance:g}")
    world = np.eye(3, 4, dtype=np.float32)
    built = gpu_ctx.set_mesh(vt.Mesh(v, f))
    tl = vt.Tlas(gpu_ctx, [(built, world)])
    assert (tl.trace_closest(_dev(far))["face"].cpu().numpy() == -1).all()
    tl.close()
    built.close()
