"""Compounds of 1 to 17 parts (the composition takes eight parts at a time, a
lane per slot of the row), internal and external ones, against the FP64 oracle,
with the bound of test_gpu_compound.py."""
import numpy as np
import pytest

import oracle as O
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import surrogate as S
from stonefish_amd import transforms as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nparts", [1, 7, 8, 9, 17])
def test_rows_of_compounds(gpu, nparts):
    print(f"case: compounds of {nparts} parts", flush=True)
    tm = M.ico_ellipsoid(0.5, 0.2, 0.2, 3)
    gm, om = H.Mesh(tm), O.Mesh.from_tri(tm)
    parts, solids = [], []
    for i in range(nparts):
        o = T.identity_gl()
        o[12:15] = [0.3 * (i % 6) - 0.75, 0.25 * (i // 6), 0.1 * (i % 3)]
        ext = i % 4 != 3
        parts.append(H.PartDesc(mesh=gm, origin=o, Cd=np.array([1.0, 0.8, 0.6]), Cf=np.array([0.1, 0.2, 0.3]),
                                external=ext, buoyant=i % 5 != 4))
        solids.append((O.make_body(om, Cd=(1.0, 0.8, 0.6), Cf=(0.1, 0.2, 0.3), volume=tm.volume(), surface=tm.area(),
                                   buoyant=i % 5 != 4), o, T.identity_gl(), ext))
    lo, hi, V, A, P = np.array([-1.3, -0.3, -0.3]), np.array([1.3, 0.8, 0.5]), 0.3, 4.0, np.array([0.0, 0.1, 0.05])
    n = 20
    batch = H.CompoundBatch([H.CompoundDesc(H.BodyDesc(mesh=None, aabb_min=lo, aabb_max=hi, volume=V, surface=A, P_CB=P),
                                            parts)] * n)
    dummy = O.Mesh(np.zeros((3, 3), np.float32), np.zeros((1, 3), np.uint32))
    comp = O.make_body(dummy, aabb_min=list(lo), aabb_max=list(hi), volume=V, surface=A, P_CB=list(P))
    rng = np.random.default_rng(nparts)
    st = np.concatenate([S.sample_states(rng, k, xy_range=(0.0, 50.0), depth_range=d)
                         for k, d in ((12, (-0.6, 0.6)), (4, (3.0, 4.0)), (4, (-4.0, -3.0)))])
    go, oo = H.Ocean(), O.Ocean()
    g = batch.compute_host(go, st)
    L, seen = 3.0, set()
    for i in range(n):
        r = O.compound_forces(comp, solids, oo, st[i, :16], st[i, 16:19], st[i, 19:22], init=np.zeros(24))
        assert g[i, 21] == r[21] and g[i, 20] == r[20], i
        seen.add(int(r[21]))
        u = np.linalg.norm(st[i, 16:19]) + np.linalg.norm(st[i, 19:22]) * L
        scale = {"b": 1000.0 * 9.81 * V * nparts, "d": 1000.0 * u ** 3 * A * nparts}
        for j in range(6):
            if (int(r[20]) >> j) & 1:
                sl = slice(3 * j, 3 * j + 3)
                bound = 1e-6 * np.linalg.norm(r[sl]) + 1e-7 * scale["b" if j < 2 else "d"] * (L if j % 2 else 1.0)
                assert np.linalg.norm(g[i, sl] - r[sl]) <= bound, (i, j, g[i, sl], r[sl])
        np.testing.assert_allclose(g[i, 18:20], r[18:20], rtol=1e-6, atol=1e-9)
    assert seen == {0, 1, 2}
