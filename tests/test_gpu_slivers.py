"""Sliver faces in large batches on waves.  A hull revolved with sin(pi) in
double precision has a ring of vertices some 1e-17 m from its pole, so the pole's
faces have |n|^2 below the smallest normal FP32 number: they are degenerate, they
are on every such hull, and they must leave the body's row as the FP64 oracle has
it.  The batches hold more than 12,288 chunks, from which on, on one layer, a
crossing chunk's whole faces come from records."""
import numpy as np
import pytest

import oracle as O
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import transforms as T
from stonefish_amd import waves as W
from util import NAMES, RTOL, STOL, bound_ratio

pytestmark = pytest.mark.gpu

BODIES, CHECKED = 12400, 48


def _sphere(radius, around, bands):
    """Rings of `around` vertices each, the poles' too: their radius is radius * sin(0)
    at one end and radius * sin(pi), not zero, at the other."""
    th = np.linspace(0.0, np.pi, bands + 1)
    ph = 2.0 * np.pi * np.arange(around) / around
    v = np.stack([radius * np.outer(np.sin(th), np.cos(ph)), radius * np.outer(np.sin(th), np.sin(ph)),
                  radius * np.outer(np.cos(th), np.ones(around))], axis=2).reshape(-1, 3)
    f = []
    for i in range(bands):
        for j in range(around):
            a, b, c, d = (i * around + j, i * around + (j + 1) % around, (i + 1) * around + j,
                          (i + 1) * around + (j + 1) % around)
            f += [[a, c, b], [c, d, b]]
    return M.TriMesh(v.astype(np.float32), np.asarray(f, np.uint32))


@pytest.mark.parametrize("K,layers", [(8, 1), (16, 1), (16, 2), (32, 1)])
def test_pole_slivers_keep_volume_and_buoyancy(gpu, K, layers):
    print(f"case: pole slivers, K {K}, {layers} layers", flush=True)
    radius, n = 0.15, 64
    tri = _sphere(radius, 32, 24)
    e1, e2 = (tri.verts[tri.faces[:, k]] - tri.verts[tri.faces[:, 0]] for k in (1, 2))
    n2 = (np.cross(e1.astype(np.float64), e2.astype(np.float64)) ** 2).sum(axis=1)
    assert ((n2 > 0) & (n2 < np.finfo(np.float32).tiny)).sum() >= 4, "faces whose |n|^2 is not a normal number"
    data = np.zeros((n, n, layers), np.float32)
    for l in range(layers):
        data[:, :, l] = W.grid_reference(W.pm_components(8, 3.0, 64.0, seed=3 + l), n)
    lengths = [64.0, 37.0][:layers]
    rgba = np.zeros((n, n, 4), np.float32)
    rgba[:, :, :layers] = data
    go = H.Ocean()
    if layers == 1:
        go.set_waves(data[:, :, 0].copy(), n, 1, lengths)
        oo = O.Ocean(wave_data=data[:, :, 0].copy(), wave_n=n, channels=1, lengths=lengths)
    else:
        go.set_waves(data, n, layers, lengths)
        oo = O.Ocean(wave_data=rgba, wave_n=n, channels=4, lengths=lengths)
    rng = np.random.default_rng(5)
    st = np.zeros((BODIES, 22))
    pos = np.stack([rng.uniform(0, 60, BODIES), rng.uniform(0, 60, BODIES), rng.uniform(-0.1, 0.1, BODIES)], axis=1)
    st[:, :16] = T.quat_to_gl(T.random_unit_quaternions(rng, BODIES), pos)
    st[:, 16:] = rng.uniform(-1, 1, (BODIES, 6))
    mesh, om = H.Mesh(tri), O.Mesh.from_tri(tri)
    batch = H.BodyBatch([H.BodyDesc(mesh=mesh, volume=0.014, surface=0.28)] * BODIES, faces_per_lane=K)
    assert batch.info()[1] > 12288
    got = batch.compute_host(go, st)
    assert np.isfinite(got).all()
    ref, ext = np.zeros((CHECKED, 24)), np.zeros((CHECKED, 22))
    ob = O.make_body(om, volume=0.014, surface=0.28)
    for i in range(CHECKED):
        ref[i], ext[i] = O.body_forces(64, ob, oo, st[i, :16], st[i, 16:19], st[i, 19:22], full=True)
    assert (ref[:, 21] == 2).sum() > CHECKED // 2, "crossing bodies"
    got = got[:CHECKED]
    assert np.array_equal(got[:, 20:22], ref[:, 20:22])
    one = np.ones((CHECKED, 3))
    worst, _ = bound_ratio(got, ref, ext, NAMES, Cd=one, Cf=0.1 * one)
    assert max(worst.values()) <= 1.0, worst
    # the error statement of tests/util.py: a face's term of the volume is at
    # most a third of its area times the hull's diameter
    wet = ref[:, 21] == 2
    bound = RTOL * ref[:, 19] + STOL * ref[:, 18] * 2.0 * radius / 3.0
    assert (np.abs(got[:, 19] - ref[:, 19])[wet] <= bound[wet]).all()
    np.testing.assert_allclose(got[:, 18], ref[:, 18], rtol=RTOL)
