"""The device traversal's own code (csrc/traverse8.h), compiled for the host, on trees of the library's
builder: node encoding and node test against the oracle's brute force at the limits of the float range."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle
import scenes
import vt

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "metal-vibe-tracer_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("traverse") / "traverse_host.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                    os.path.join(HERE, "traverse_host.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def trace(lib, v, f, rays):
    nodes, tris, _, root = vt.build_bvh8_host(vt.Mesh(v, f))
    rays = np.ascontiguousarray(rays, np.float32)
    n = rays.shape[1]
    out = {k: np.empty(n, np.float32) for k in ("t", "b1", "b2")}
    out["face"], out["occluded"], out["visits"] = np.empty(n, np.int32), np.empty(n, np.uint8), np.empty(2, np.uint64)
    lib.closest(_ptr(nodes), ctypes.c_uint32(len(nodes)), _ptr(tris), ctypes.c_float(root), _ptr(rays), ctypes.c_uint32(n),
                *[_ptr(a) for a in out.values()])
    return out


def check(lib, v, f, rays):
    got, ref = trace(lib, v, f, rays), oracle.Scene(v, f, with_bvh=False).closest(rays, mode=1)
    for k in ("t", "b1", "b2", "face"):
        same = (got[k] == ref[k]) | (np.isnan(got[k]) & np.isnan(ref[k]))
        assert same.all(), f"{k}: {int((~same).sum())} of {rays.shape[1]} rays differ"
    assert np.array_equal(got["occluded"] != 0, ref["face"] >= 0)
    return got, ref


def test_ordinary_scene(lib):
    v, f = scenes.scattered_triangles(500, seed=2)
    check(lib, v, f, np.concatenate([scenes.random_rays(3000, 1), scenes.axis_rays(500, 1)], axis=1))


# Either side of the size from which node boxes are scaled (2^82 = 4.8e24), where a grid step times 2^24
# and 1e8 would overflow (5e25), and where the step itself would.
LENGTHS = [1e6, 4.7e24, 4.9e24, 1e25, 1e26, 1e28, 1e32, 1e37]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("length", LENGTHS)
def test_long_strips(lib, length, axis):
    v, f, rays = scenes.long_strip(length, axis)
    _, ref = check(lib, v, f, rays)
    assert (ref["face"][:64] >= 0).all()


@pytest.mark.parametrize("extents", [(30, -12, -5), (-17, -3, 26), (31, -4, 0), (5, -13, 32), (24, 2, 1), (17, 18, 6)])
def test_uneven_extents(lib, extents):
    rng = np.random.default_rng(7)
    scale = 10.0 ** np.array(extents, np.float64)
    tri = (rng.uniform(-0.9, 0.9, (300, 1, 3)) + rng.uniform(-0.2, 0.2, (300, 3, 3))) * scale
    v, f = scenes.mesh_from_triangles(tri.astype(np.float32))
    rays = np.concatenate([scenes.random_rays(3000, 3), scenes.axis_rays(1000, 3)], axis=1)
    rays[0:3] *= scale[:, None].astype(np.float32)
    for along in (False, True):
        if along:
            rays[3:6] *= scale[:, None].astype(np.float32)
        check(lib, v, f, rays)


@pytest.mark.parametrize("distance", [1e30, 2.8e36, 3e36, 1e37, 3.4e38])
def test_far_origins_enter_nothing(lib, distance):
    # From 2.9e36 on e / |direction| overflows for parallel axes.  No ray gets past the root node.
    v, f = scenes.scattered_triangles(500, seed=2)
    rays = scenes.far_rays(distance)
    got, ref = check(lib, v, f, rays)
    assert (ref["face"] < 0).all()
    assert got["visits"].tolist() == [rays.shape[1], 0]
