"""GPU tests of the wavefront's queues at the sizes where their block-wide appends can go wrong: path
counts around a wave (64), a block (256) and several blocks, against the reference integrator restated
in the oracle, and the cache's query and record counts against the rule that picks training paths."""
import numpy as np
import pytest

import oracle
import scenes
import vt

pytestmark = pytest.mark.gpu

MATS = [dict(type=0, albedo=(0.73, 0.73, 0.73)), dict(type=0, albedo=(0.65, 0.05, 0.05)),
        dict(type=0, albedo=(0.12, 0.45, 0.15)), dict(type=3, albedo=(0, 0, 0), emission=(17, 17, 17))]
TARGET = (0.0, -0.1, 0.0)


@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (7, 9, 1), (64, 1, 1), (65, 1, 1), (51, 5, 1), (256, 1, 1), (257, 1, 1),
                                     (33, 31, 5), (128, 96, 3)])
def test_images_at_block_edges(gpu_ctx, w, h, spp):
    # Lost, doubled or misplaced paths change whole pixels.  Up to 3% of the pixels may differ beyond
    # rounding (the integrator's parity bar: a path whose transcendentals round another way can meet
    # another triangle), and at least one.
    mesh = vt.cornell()
    scene = gpu_ctx.set_mesh(mesh)
    scene.set_materials(vt.cornell_materials(17.0))
    r = vt.Renderer(gpu_ctx)
    print(f"cornell {w}x{h} {spp} spp", flush=True)
    r.render(scene, w, h, vt.orbit_eye(), TARGET, 42.0, max_depth=6, samples=spp, sample_index=1)
    got = r.readback()[..., :3].astype(np.float64)
    r.close()
    scene.close()
    frame = dict(width=w, height=h, eye=vt.orbit_eye(), target=TARGET, fov=42.0, max_depth=6)
    ref = oracle.render(oracle.Scene(mesh.vertices, mesh.faces), MATS, frame, 1, spp, precision="f32").reshape(h, w, 3)
    bad = (~np.isclose(got, ref, rtol=1e-3, atol=1e-4).all(axis=2)).sum()
    assert bad <= max(1, int(0.03 * w * h)), bad


def _pcg(v):
    v = np.asarray(v, np.uint64) & 0xffffffff
    s = (v * 747796405 + 2891336453) & 0xffffffff
    w = (((s >> ((s >> 28) + 4)) ^ s) * 277803737) & 0xffffffff
    return (w >> 22) ^ w


@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (19, 14), (97, 61)])
def test_record_counts(gpu_ctx, w, h):
    # The training paths that scatter to a second non-emissive surface leave one record each, so the
    # records cannot exceed the paths the hash picks.  The box (2 units wide, 3.4 away at a 42 degree
    # view 2.6 units high) covers at least 0.59 / aspect >= 0.37 of these images and a path that enters
    # it rarely ends or leaves at once, so at least a quarter of the picked paths leave a record.
    mesh = vt.cornell()
    scene = gpu_ctx.set_mesh(mesh)
    scene.set_materials(vt.cornell_materials(17.0))
    cache, r = vt.NRC(gpu_ctx, seed=2), vt.Renderer(gpu_ctx)
    r.set_cache(cache)
    r.render(scene, w, h, vt.orbit_eye(), TARGET, 42.0, max_depth=4, samples=1, sample_index=3, cache=2, train_period=2)
    x, t, made = r.cache_records()
    pix = np.arange(w * h, dtype=np.uint64)
    key = _pcg((pix * 0x9E3779B9 & 0xffffffff) ^ ((3 * 0x85EBCA6B) & 0xffffffff))
    picked = int((key % 2 == 0).sum())
    print(f"{w}x{h}: {made} records of {picked} training paths", flush=True)
    assert made == len(x) <= picked and np.isfinite(t).all()
    assert ((x >= 0) & (x <= 1)).all()
    if picked > 100:
        assert made > 0.25 * picked
        assert len(np.unique(x.view(np.uint32), axis=0)) == made   # no record twice
    r.close()
    scene.close()
    cache.close()


@pytest.mark.parametrize("w,h", [(1, 1), (16, 16), (257, 1), (64, 32), (2049, 1), (73, 61)])
@pytest.mark.parametrize("mode", [0, 1])
def test_material_order_changes_nothing(gpu_ctx, w, h, mode):
    # Frames below 2^16 paths are shaded in queue order by default, in the order of their shading class on
    # request: the same image, bit for bit, around the 2048 paths a block lists at a time.
    mesh, mats = scenes.materials_cornell("opaque")
    scene = gpu_ctx.set_mesh(mesh)
    scene.set_materials(scenes.vt_materials(mats))
    imgs = []
    for sort in (False, True):
        r = vt.Renderer(gpu_ctx)
        r.render(scene, w, h, vt.orbit_eye(), TARGET, 42.0, max_depth=5, samples=2, sample_index=1, sampling_mode=mode,
                 material_sort=sort)
        imgs.append(r.readback())
        r.close()
    scene.close()
    print(f"{w}x{h} mode {mode}: mean {imgs[0][..., :3].mean():.6f}", flush=True)
    assert np.array_equal(imgs[0], imgs[1])


@pytest.mark.parametrize("w,h", [(1, 1), (16, 16), (257, 1), (33, 17)])
def test_restir_lists_every_diffuse_pixel(gpu_ctx, w, h):
    # ReSTIR's first pass runs over a list of the diffuse pixels: around a block of 256, against the oracle
    # (up to 5% of the pixels may differ beyond rounding, the materials' ReSTIR parity bar, at least one).
    mesh, mats = scenes.materials_cornell("opaque")
    scene = gpu_ctx.set_mesh(mesh)
    scene.set_materials(scenes.vt_materials(mats))
    r = vt.Renderer(gpu_ctx)
    r.render(scene, w, h, vt.orbit_eye(), TARGET, 42.0, max_depth=3, samples=2, sample_index=1, sampling_mode=0,
             indirect_reuse=1)
    got = r.readback()[..., :3].astype(np.float64)
    r.close()
    scene.close()
    frame = dict(width=w, height=h, eye=vt.orbit_eye(), target=TARGET, fov=42.0, max_depth=3, indirect_reuse=1)
    ref = oracle.render_restir(oracle.Scene(mesh.vertices, mesh.faces), mats, frame, 1, 2, candidates=4).reshape(h, w, 3)
    bad = (~np.isclose(got, ref, rtol=1e-3, atol=1e-4).all(axis=2)).sum()
    print(f"restir {w}x{h}: {bad} pixels differ", flush=True)
    assert bad <= max(1, int(0.05 * w * h))
