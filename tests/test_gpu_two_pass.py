"""Large batches on waves, where the face launch takes a crossing chunk's rows
twice (more than 12,288 chunks, 8 faces per lane or more, one layer; on two layers
once): from face records, and from packed faces and vertices where the batch's
distinct meshes hold more than two million faces.  Meshes of one face, of a row of 64, of
a chunk with one face more or less, and shuffled ones, whose vertex windows are
too large to stage and whose batches take the rows once.  Every body's row is held to the FP64 oracle with the error
statement of tests/util.py, and does not depend on the launch's shape."""
from functools import lru_cache

import numpy as np
import pytest

import oracle as O
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import transforms as T
from stonefish_amd import waves as W
from util import NAMES, RTOL, STOL, bound_ratio

pytestmark = pytest.mark.gpu

SIZES = (1, 63, 64, 65, 511, 513, 1023, 1025, 2047, 2049, 4096 + 65)
COPIES = 900   # 12,600 chunks at 32 faces per lane
CHUNKS, RADIUS = 12288, 1.1


def _tris(shuffle):
    hull = M.ico_ellipsoid(RADIUS, 0.5, 0.4, 5)
    tris = []
    for i, m in enumerate(SIZES):
        f = hull.faces[2000 * (i % 3):][:m]
        if shuffle:
            f = hull.faces[np.random.default_rng(i).permutation(len(hull.faces))[:m]]
        tris.append(M.TriMesh(hull.verts, np.ascontiguousarray(f)))
    return hull, tris


def _states(n):
    rng = np.random.default_rng(11)
    s = np.zeros((n, 22))
    pos = np.stack([rng.uniform(0, 60, n), rng.uniform(0, 60, n), rng.uniform(-0.8, 1.2, n)], axis=1)
    s[:, :16] = T.quat_to_gl(T.random_unit_quaternions(rng, n), pos)
    s[:, 16:19] = rng.uniform(-2, 2, (n, 3))
    s[:, 19:22] = rng.uniform(-1, 1, (n, 3))
    return s


def _sea(layers):
    n, lengths = 64, [64.0, 37.0][:layers]
    data = np.zeros((n, n, layers), np.float32)
    for l in range(layers):
        data[:, :, l] = W.grid_reference(W.pm_components(8, 5.0, 64.0, seed=3 + l), n)
    go = H.Ocean()
    if layers == 1:
        go.set_waves(data[:, :, 0].copy(), n, 1, lengths)
        return go, O.Ocean(wave_data=data[:, :, 0].copy(), wave_n=n, channels=1, lengths=lengths)
    go.set_waves(data, n, layers, lengths)
    rgba = np.zeros((n, n, 4), np.float32)
    rgba[:, :, :2] = data
    return go, O.Ocean(wave_data=rgba, wave_n=n, channels=4, lengths=lengths)


@lru_cache(maxsize=3)
def _reference(layers, shuffle):
    _, tris = _tris(shuffle)
    st, oo = _states(len(tris) * COPIES), _sea(layers)[1]
    bodies = [O.make_body(O.Mesh.from_tri(t), volume=0.2, surface=1.0) for t in tris]
    ref, ext = np.zeros((len(st), 24)), np.zeros((len(st), 22))
    for i, s in enumerate(st):
        ref[i], ext[i] = O.body_forces(64, bodies[i % len(tris)], oo, s[:16], s[16:19], s[19:22], full=True)
    return ref, ext


@pytest.mark.parametrize("K", [8, 16, 32])
@pytest.mark.parametrize("layers,shuffle,faces", [(1, False, "records"), (2, False, "records"), (1, True, "records"),
                                                  (1, False, "packed"), (2, False, "packed")])
def test_two_pass_rows_match_the_oracle(gpu, K, layers, shuffle, faces):
    print(f"case: K {K}, {layers} layers, shuffled {shuffle}, {faces}", flush=True)
    hull, tris = _tris(shuffle)
    meshes = [H.Mesh(t) for t in tris]
    descs = [H.BodyDesc(mesh=m, volume=0.2, surface=1.0) for _ in range(COPIES) for m in meshes]
    n = len(descs)
    if faces == "packed":
        descs += [H.BodyDesc(mesh=H.Mesh(hull), volume=0.2, surface=1.0) for _ in range(100)]
    st = _states(n)
    st = np.concatenate([st, st[:len(descs) - n]])
    go, _ = _sea(layers)
    batch = H.BodyBatch(descs, faces_per_lane=K)
    assert batch.info()[1] > CHUNKS
    assert (sum(m.nf for m in meshes) + 20480 * (len(descs) - n) > 2_000_000) == (faces == "packed")
    got = batch.compute_host(go, st)
    batch.set_opts(faces_per_lane=K, waves=700, split_passes=1)
    again = batch.compute_host(go, st)
    assert np.array_equal(got, again), "rows depend on the launch's shape"
    got = got[:n]
    ref, ext = _reference(layers, shuffle)
    assert {0.0, 1.0, 2.0} <= set(ref[:, 21])
    assert np.array_equal(got[:, 20:22], ref[:, 20:22])
    one = np.ones((n, 3))
    worst, _ = bound_ratio(got, ref, ext, NAMES, Cd=one, Cf=0.1 * one)
    assert max(worst.values()) <= 1.0, worst
    np.testing.assert_allclose(got[:, 18], ref[:, 18], rtol=RTOL, atol=1e-9)
    # a face's term of the volume is at most a third of its area times its
    # distance from the point below the body's centre, 3 m here
    wet = ref[:, 20].astype(int) & 128 > 0
    assert (np.abs(got[:, 19] - ref[:, 19])[wet] <= (RTOL * np.abs(ref[:, 19]) + STOL * ref[:, 18])[wet]).all()
