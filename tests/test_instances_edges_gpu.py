"""GPU tests of the two-level traversal at its edges: ray counts around a wave and a block, hierarchies of
growing depth on both levels, mirrored coincident instances whose hits tie at face 0 with other
barycentrics, and rays with NaN and exact limits, against the two-level oracle bit for bit."""
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


def _check(ctx, meshes, inst, rays, what):
    import torch
    built = [ctx.set_mesh(vt.Mesh(v, f)) for v, f in meshes]
    tl = vt.Tlas(ctx, [(built[a], w) for a, w in inst])
    got = {k: x.cpu().numpy() for k, x in tl.trace_closest(_dev(rays)).items()}
    occ = tl.trace_any(_dev(rays)).cpu().numpy()
    torch.cuda.synchronize()
    info = tl.info
    ref = oinst.closest([oracle.Scene(v, f, with_bvh=False) for v, f in meshes], inst, rays)
    print(f"{what}: {info}, {rays.shape[1]} rays, {int((ref['face'] >= 0).sum())} hits", flush=True)
    got["instance"] = got["instance"].view(np.uint32)
    ref["instance"] = ref["instance"].astype(np.uint32)
    for k in ("t", "b1", "b2", "face", "instance"):
        same = (got[k] == ref[k]) | (np.isnan(got[k]) & np.isnan(ref[k]))
        assert same.all(), f"{what}: {k} differs at {np.nonzero(~same)[0][:5]}"
    assert np.array_equal(occ != 0, ref["face"] >= 0), what
    ctx.check()
    tl.close()
    for s in built:
        s.close()
    return info, ref


def _world(scale, at):
    w = np.zeros((3, 4), np.float32)
    w[:, :3] = np.eye(3) * scale
    w[:, 3] = at
    return w


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 16385, 131073])
def test_ray_counts(gpu_ctx, n):
    v, f = scenes.scattered_triangles(40, seed=3)
    rng = np.random.default_rng(1)
    inst = [(0, _world(rng.uniform(0.2, 1.0), rng.uniform(-1, 1, 3))) for _ in range(11)]
    _check(gpu_ctx, [(v, f)], inst, scenes.random_rays(n, n), f"{n} rays")


@pytest.mark.parametrize("triangles,instances", [(1, 1), (1, 300), (60, 8), (60, 60), (150, 9), (150, 150), (400, 300)])
def test_depths(gpu_ctx, triangles, instances):
    # Triangles and instances along geometric series: the surface-area splits peel them off a few at a
    # time, so the hierarchies are as deep as their counts allow.
    s = 0.8 ** np.arange(triangles)
    tri = np.stack([np.stack([s, s, 0 * s], 1), np.stack([1.2 * s, s, 0.1 * s], 1), np.stack([s, 1.2 * s, 0.1 * s], 1)], 1)
    v, f = scenes.mesh_from_triangles(tri.astype(np.float32))
    at = 0.8 ** np.arange(instances)
    inst = [(0, _world(max(0.3 * a, 1e-5), (2 * a - 1, -a, 0.5 * a))) for a in at]
    rng = np.random.default_rng(2)
    n = 8000
    # Aimed at points of the series on both levels, in log scale, from random origins.
    k, j = rng.integers(0, instances, n), rng.integers(0, triangles, n)
    w = np.stack([x[1] for x in inst])[k].astype(np.float64)
    bary = rng.dirichlet((1, 1, 1), n)
    p = np.einsum("nij,nj->ni", w[:, :, :3], np.einsum("nk,nkj->nj", bary, tri[j])) + w[:, :, 3]
    o = p + rng.normal(size=(n, 3)) * (10.0 ** rng.uniform(-3, 0.5, n))[:, None]
    d = p - o
    rays = np.concatenate([o.T, (d / np.linalg.norm(d, axis=1, keepdims=True)).T, np.zeros((1, n)), np.full((1, n), 1e30)])
    info, ref = _check(gpu_ctx, [(v, f)], inst, rays.astype(np.float32), f"{triangles} x {instances}")
    # Triangles below 2^-24 of the origins' distance cannot be aimed at in float32; the larger ones are hit.
    assert (ref["face"] >= 0).sum() > 500


@pytest.mark.parametrize("order", [(0, 1), (1, 0), (0, 1, 0, 1, 1), (1, 1, 0)])
def test_ties_of_mirrored_instances(gpu_ctx, order):
    # One triangle, as it is and with x and y exchanged: the same points, met at the same t, with b1 and
    # b2 exchanged; the smaller instance index keeps the hit whatever order they are visited in.
    v, f = scenes.mesh_from_triangles(np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]], np.float32))
    same = _world(1.0, 0.0)
    swapped = same[[1, 0, 2]]
    rng = np.random.default_rng(6)
    n = 3000
    rays = np.zeros((8, n), np.float32)
    rays[0:2] = rng.integers(0, 256, (2, n)) / np.float32(256)
    rays[2] = 1.0
    rays[5] = -1.0
    rays[7] = 100.0
    rays[7, 1::3] = 1.0      # ends exactly at the triangle
    rays[7, 2::30] = np.nan  # nothing is nearer than a NaN
    _check(gpu_ctx, [(v, f)], [(0, (same, swapped)[o]) for o in order], rays, f"order {order}")
