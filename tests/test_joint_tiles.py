"""A joint step of a tiled model (nimblesm_amd/csrc/nsm_tiled.hip) keeps u and
v of the boundary nodes in arrays that hold those nodes' rows only: on the
CPU, that every row it reads from them is theirs, on meshes of separate
bodies too, where a tile may hold no boundary node; on the device, that such
meshes advance to the bits of separate launches."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import nimblesm_amd as N
from oracle import oracle as O

from test_tiles import ROOT, build, check_invariants


@pytest.fixture(scope="module")
def joint_lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("joint") / "libjoint.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out,
                    os.path.join(ROOT, "tests", "joint_tiles_shim.cpp"),
                    os.path.join(ROOT, "nimblesm_amd", "csrc", "nsm_tiles.cpp")], check=True)
    lib = C.CDLL(out)
    lib.tiles_build.restype = C.c_void_p
    lib.tiles_build.argtypes = [C.c_int64, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_int]
    lib.tiles_sizes.argtypes = [C.c_void_p, C.c_void_p]
    lib.tiles_copy.argtypes = [C.c_void_p] + [C.c_void_p] * 15
    lib.tiles_staged.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    lib.tiles_free.argtypes = [C.c_void_p]
    return lib


def bodies(sizes):
    """Separate cubes of sizes[b]^3 elements, a block each, and its first element."""
    X, conn, off = [], [], [0]
    nodes = 0
    for b, n in enumerate(sizes):
        x, c = O.jittered_cube(n, 5 + b, 0.1)
        X.append(x * n / max(sizes) + [2.0 * b, 0.0, 0.0])
        conn.append(c + nodes)
        nodes += len(x)
        off.append(off[-1] + len(c))
    return np.vstack(X), np.vstack(conn).astype(np.int32), np.array(off)


SIZES = [(2, 12), (12, 2), (12, 2, 11), (1, 10, 2, 1), (3, 3, 9), (12,)]


@pytest.mark.parametrize("tile", [64, 128, 256, 512])
@pytest.mark.parametrize("sizes", SIZES)
def test_boundary_rows_are_boundary_nodes(joint_lib, sizes, tile):
    X, conn, off = bodies(sizes)
    t = build(joint_lib, X, conn, off, tile)
    check_invariants(t, len(X), conn, off)
    lib, no = joint_lib, t["node_off"]
    h = lib.tiles_build(len(X), X.ctypes.data, conn.ctypes.data, len(off) - 1, off.ctypes.data, tile)
    bnd = np.zeros(len(X), bool)
    bnd[t["bnd_nodes"]] = True
    alone = 0
    for k in range(len(no) - 1):
        ids, row = np.zeros(2 * tile, np.int32), np.zeros(2 * tile, np.uint8)
        lib.tiles_staged(h, k, ids.ctypes.data, row.ctypes.data)
        nn = no[k + 1] - no[k]
        assert np.array_equal(ids[:nn], t["nodes"][no[k]:no[k + 1]]) and np.all(ids[nn:] == ids[nn - 1])
        assert np.array_equal(row != 0, bnd[ids])
        alone += not bnd[ids].any()
    lib.tiles_free(h)
    assert alone >= sum(n ** 3 <= tile for n in sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,tile", [((2, 12), 128), ((12, 2, 11), 64), ((1, 10, 2, 1), 256), ((3, 12), 512)])
def test_separate_bodies_match_separate_launches(hip_device, monkeypatch, sizes, tile):
    """Bodies that fill one tile and less beside one of several tiles: the
    joint launches run (their second buffers are there) and give the bits of
    the element and node launches, which kernel timing asks for."""
    monkeypatch.setenv("NSM_TILE_ELEMS", str(tile))
    X, conn, off = bodies(sizes)
    blocks = [N.Block(b + 1, conn[off[b]:off[b + 1]], N.NeohookeanMaterial.from_young(7800.0, 200e9 / (b + 1), 0.3))
              for b in range(len(sizes))]
    bottom, top = (np.nonzero(X[:, 2] == z)[0].astype(np.int32) for z in (0.0, 1.0))
    got = []
    for separate in (False, True):
        m = N.ModelData(X, blocks, precision="mixed")
        m.AddBoundaryCondition("prescribed_velocity", bottom, 2, 0.0)
        m.AddBoundaryCondition("initial_velocity", top, 0, 2.0)
        m.SetReactionNodes(bottom, 2)
        m.ComputeLumpedMass()
        dt = 0.5 * m.GetCriticalTimeStep()
        m.ApplyInitialConditions()
        m.SetVectorNodeData("displacement", 1e-3 * np.sin(3 * X) * X[:, 2:3])
        if separate:
            m.EnableKernelTiming(True, every=1000)
        before, t, out = m.Info()["device_bytes"], 0.0, []
        for a, b in ((0, 3), (3, 7), (7, 16)):
            t = m.ExplicitSteps(a, b, 16, 4, dt, t)
            if a == 0:
                assert (m.Info()["device_bytes"] > before) == (not separate)
            out += [m.GetVectorNodeData(f) for f in ("displacement", "velocity", "acceleration", "internal_force")]
            out += [m.GetIntegrationPointData("stress"), m.GetReactionHistory(0, b)]
        got.append(out)
        m.close()
    assert np.linalg.norm(got[0][-1]) > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,n", [("fp64", 1), ("fp64", 5), ("mixed", 5)])
def test_second_buffers_in_used_memory(hip_device, monkeypatch, precision, n):
    """The buffers of the joint launches may lie where other data was: models
    made after memory full of NaN has been given back advance to the bits of
    separate launches."""
    import torch

    monkeypatch.setenv("NSM_TILE_ELEMS", "64")
    X, conn, _ = bodies((n,))
    got = []
    for separate in (False, True):
        m = N.ModelData(X, [N.Block(1, conn, N.NeohookeanMaterial.from_young(7800.0, 200e9, 0.3))], precision=precision)
        m.ComputeLumpedMass()
        dt = 0.5 * m.GetCriticalTimeStep()
        m.SetVectorNodeData("displacement", 1e-3 * np.sin(3 * X) * X[:, 2:3])
        if separate:
            m.EnableKernelTiming(True, every=1000)
        used = [torch.full((k,), float("nan"), device=hip_device) for k in (1 << 10, 1 << 14, 1 << 18, 1 << 22)]
        torch.cuda.synchronize()
        del used
        torch.cuda.empty_cache()
        before = m.Info()["device_bytes"]
        m.ExplicitSteps(0, 5, 5, 0, dt, 0.0)
        assert (m.Info()["device_bytes"] > before) == (not separate)
        got.append([m.GetVectorNodeData(f) for f in ("displacement", "velocity", "acceleration", "internal_force")])
        m.close()
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
