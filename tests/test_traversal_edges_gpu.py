"""GPU tests of the traversal at the edges of its node encoding and of how rays are dealt to waves:
meshes from one triangle up (every filling of a node's eight slots and three-triangle leaves), scenes far
from the origin and very small or flat ones, ray counts around a wave's 64 and a block's 512, rays that
end exactly at a hit and rays with a NaN limit, against the oracle's brute force, bit for bit."""
import numpy as np
import pytest

import oracle
import scenes
import vt

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda:0")


def _triangles(n, seed):
    """Random triangles of about half the size of the box the rays start in."""
    rng = np.random.default_rng(seed)
    c, e = rng.uniform(-0.9, 0.9, (n, 1, 3)), rng.uniform(-0.5, 0.5, (n, 3, 3))
    return scenes.mesh_from_triangles((c + e).astype(np.float32))


def _check(ctx, v, f, rays, what):
    import torch
    scene = ctx.set_mesh(vt.Mesh(v, f))
    h = {k: x.cpu().numpy() for k, x in scene.trace_closest(_dev(rays)).items()}
    occ = scene.trace_any(_dev(rays)).cpu().numpy()
    torch.cuda.synchronize()
    ref = oracle.Scene(v, f, with_bvh=False).closest(rays, mode=1)
    print(f"{what}: {len(f)} triangles, {rays.shape[1]} rays, {int((ref['face'] >= 0).sum())} hits", flush=True)
    for k in ("t", "b1", "b2", "face"):
        same = (h[k] == ref[k]) | (np.isnan(h[k]) & np.isnan(ref[k]))
        assert same.all(), f"{what}: {k} differs at {np.nonzero(~same)[0][:5]}"
    assert np.array_equal(occ != 0, ref["face"] >= 0), what
    scene.close()


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 9, 23, 24, 25, 26, 60, 200])
def test_node_fillings(gpu_ctx, count):
    v, f = _triangles(count, seed=count)
    rays = np.concatenate([scenes.random_rays(6000, count), scenes.axis_rays(600, count)], axis=1)
    _check(gpu_ctx, v, f, rays, f"scattered {count}")


@pytest.mark.parametrize("scale,shift", [(1.0, (4000.0, -3000.0, 5000.0)), (1e-6, (0.0, 0.0, 0.0)), (1e6, (0.0, 0.0, 0.0)),
                                         ((1.0, 0.0, 1.0), (0.0, 0.25, 0.0))])
def test_scales_and_places(gpu_ctx, scale, shift):
    # Steps of the node grid from 2^-28 to 2^14, a zero extent along y, and an origin far from the scene.
    v, f = _triangles(300, seed=9)
    v = v.copy()
    v[:, :3] = (v[:, :3].astype(np.float64) * scale + shift).astype(np.float32)
    rays = scenes.random_rays(8000, 4)
    rays[0:3] = (rays[0:3].astype(np.float64) * np.max(scale) + np.array(shift)[:, None]).astype(np.float32)
    _check(gpu_ctx, v, f, rays, f"scale {scale} shift {shift}")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 16384, 16385, 131073])
def test_ray_counts(gpu_ctx, n):
    v, f = _triangles(40, seed=3)
    _check(gpu_ctx, v, f, scenes.random_rays(n, n), f"{n} rays")


def test_ray_limits(gpu_ctx):
    # [tmin, tmax): a limit exactly at the hit excludes it, the next float includes it; a NaN limit is a miss.
    v, f = _triangles(200, seed=6)
    rays = scenes.random_rays(8000, 8)
    ref = oracle.Scene(v, f, with_bvh=False).closest(rays, mode=1)
    hit = ref["face"] >= 0
    rays = np.ascontiguousarray(rays[:, hit])
    t = ref["t"][hit].astype(np.float32)
    for tmax in (t, np.nextafter(t, np.float32(np.inf)), np.zeros_like(t), np.full_like(t, np.inf)):
        r = rays.copy()
        r[7] = tmax
        _check(gpu_ctx, v, f, r, "tmax")
    r = rays.copy()
    r[6] = t
    _check(gpu_ctx, v, f, r, "tmin at the hit")
    r = rays.copy()
    r[7] = np.nan
    scene = gpu_ctx.set_mesh(vt.Mesh(v, f))
    h = scene.trace_closest(_dev(r))
    assert (h["face"].cpu().numpy() == -1).all() and np.isnan(h["t"].cpu().numpy()).all()
    assert (h["b1"].cpu().numpy() == 0).all()
    assert (scene.trace_any(_dev(r)).cpu().numpy() == 0).all()
    scene.close()


@pytest.mark.parametrize("count,nodes", [(640, 63), (624, 64), (660, 65), (716, 67)])
def test_where_nodes_are_encoded(gpu_ctx, count, nodes):
    # Up to 64 nodes are encoded by the host, more by a kernel.
    v, f = scenes.scattered_triangles(count, seed=1)
    assert len(vt.build_bvh8_host(vt.Mesh(v, f))[0]) == nodes
    rays = np.concatenate([scenes.random_rays(6000, count), scenes.axis_rays(600, count)], axis=1)
    _check(gpu_ctx, v, f, rays, f"{nodes} nodes")
