"""A varying current or wind is sampled at a whole face's centroid in FP64.  Near
the wall of a pipe with an exponent below 1 its velocity (1 - d/r)^gamma is steep:
at 1e-7 of the radius from the wall a centroid off by 1e-8 m moves it by a
per cent.  Triangles of some metres, each with its centroid there, are held to
the FP64 oracle with the error statement of tests/util.py: the per-body call,
the one-launch step and the face launch, in the water and in the wind."""
import numpy as np
import pytest

import oracle as O
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from util import bound_ratio

pytestmark = pytest.mark.gpu

N = 24


def _case(i):
    """A triangle and the pipe along z whose wall its centroid is at."""
    rng = np.random.default_rng(100 + i)
    p = rng.uniform(-1.9, 1.9, (3, 3)).astype(np.float32)
    c = p.astype(np.float64).sum(axis=0) / 3.0
    d = (1.0 - 1e-7) * (np.array([1.0, 0.0]) if i % 2 else np.array([0.0, 1.0]))
    return M.TriMesh(p, np.array([[0, 1, 2]], np.uint32)), np.array([c[0] - d[0], c[1] - d[1]])


def _pose(z):
    t = np.zeros(16)
    t[[0, 5, 10, 15]] = 1.0
    t[14] = z
    return t


def _pipe(axis, z):
    return [axis[0], axis[1], z - 10.0], [axis[0], axis[1], z + 10.0], 1.0, 1.0, 2.0, 0.1


@pytest.mark.parametrize("path", ["call", "step", "faces"])
def test_current_at_the_exact_centroid(gpu, path):
    print(f"case: current at the centroid, {path}", flush=True)
    zero = np.zeros(3)
    got, ref, ext = np.zeros((N, 24)), np.zeros((N, 24)), np.zeros((N, 22))
    for i in range(N):
        tri, axis = _case(i)
        mesh, om, T = H.Mesh(tri), O.Mesh.from_tri(tri), _pose(20.0)
        a, b, r1, r2, vin, gamma = _pipe(axis, 20.0)
        go = H.Ocean()
        go.add_pipe(a, b, r1, r2, vin, gamma)
        go.enable_currents(True)
        oo = O.Ocean(currents=[(2, 1, a + [0.0, 0.0, 1.0, 20.0, r1, r2, vin, gamma])], currents_enabled=True)
        if path == "call":
            out = np.zeros((4, 3))
            H.ComputeHydrodynamicForcesSubmerged(mesh, go, T, T, zero, zero, *out)
            got[i, 6:18] = out.ravel()
            ref[i], ext[i] = O.submerged(64, om, oo, T, T, zero, zero, full=True)
            ref[i, 20] = 60
        else:
            batch = H.BodyBatch([H.BodyDesc(mesh=mesh)], faces_per_lane=16, split_passes=int(path == "faces"))
            got[i] = batch.compute_host(go, np.concatenate([T, zero, zero])[None])[0]
            ref[i], ext[i] = O.body_forces(64, O.make_body(om), oo, T, zero, zero, full=True)
            assert got[i, 21] == ref[i, 21] == 1.0
    names = ("Fdq", "Tdq", "Fdf", "Tdf")
    kw = {} if path == "call" else dict(Cd=np.ones((N, 3)), Cf=np.full((N, 3), 0.1))
    assert np.abs(ref[:, 12:15]).max(axis=1).min() > 0
    worst, _ = bound_ratio(got, ref, ext, names, **kw)
    assert max(worst.values()) <= 1.0, worst


def test_wind_at_the_exact_centroid(gpu):
    print("case: wind at the centroid", flush=True)
    zero = np.zeros(3)
    for i in range(N):
        tri, axis = _case(i)
        mesh, om, T = H.Mesh(tri), O.Mesh.from_tri(tri), _pose(-20.0)
        a, b, r1, r2, vin, gamma = _pipe(axis, -20.0)
        atm = H.Atmosphere()
        atm.add_pipe(a, b, r1, r2, vin, gamma)
        F, Tq = np.zeros(3), np.zeros(3)
        H.ComputeAerodynamicForces(mesh, atm, T, T, zero, zero, F, Tq)
        wind = [(2, a + [0.0, 0.0, 1.0, 20.0, r1, r2, vin, gamma])]
        rF, rT = O.aero(om, 1.225, wind, T, T, zero, zero)[:2]
        # one face: no cancellation but in its lever arm, 2 m at most
        assert np.linalg.norm(F - rF) <= 1.2e-6 * np.linalg.norm(rF)
        assert np.linalg.norm(Tq - rT) <= 1.2e-6 * 2.0 * np.linalg.norm(rF)
