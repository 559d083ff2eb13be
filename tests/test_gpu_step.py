"""The one-launch step of small batches and of the per-body calls, at the
sizes where it can go wrong: chunks of one face, of a whole row of 64 and of
a whole chunk with one face more or less, bodies of one and of several chunks,
vertex windows too large to stage, masks, bodies without face work.

A batch's rows are held to those of the general path (prologue, face launches,
epilogue; split_passes = 1 selects it) bit for bit; the per-body calls to the
FP64 oracle with the error statement of tests/util.py."""
import numpy as np
import pytest

import oracle as O
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import transforms as T
from stonefish_amd import waves as W
from util import bound_ratio

pytestmark = pytest.mark.gpu


def _part(tm, m, shuffle=False):
    """The first m faces of a mesh (any set of faces is a valid input)."""
    f = tm.faces[:m]
    if shuffle:
        f = f[np.random.default_rng(3).permutation(len(f))]
    return M.TriMesh(tm.verts, np.ascontiguousarray(f))


def _ocean(sea, jet):
    o = H.Ocean()
    if sea:
        n, layers = sea
        data = np.zeros((n, n, layers), np.float32)
        for l in range(layers):
            data[:, :, l] = W.grid_reference(W.pm_components(8, 5.0, 64.0, seed=3 + l), n)
        o.set_waves(data, n, layers, [64.0, 37.0][:layers])
    if jet:
        o.add_jet((30.0, 30.0, 0.5), (0.6, 0.8, 0.0), 30.0, 2.0)
        o.add_uniform_current((0.3, -0.2, 0.0))
        o.enable_currents(True)
    return o


def _states(rng, n, depth=(-1.2, 1.8)):
    s = np.zeros((n, 22))
    pos = np.stack([rng.uniform(0, 60, n), rng.uniform(0, 60, n), rng.uniform(*depth, n)], axis=1)
    s[:, :16] = T.quat_to_gl(T.random_unit_quaternions(rng, n), pos)
    s[:, 16:19] = rng.uniform(-2, 2, (n, 3))
    s[:, 19:22] = rng.uniform(-1, 1, (n, 3))
    return s


def _same_bits(a, b, what):
    assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), what


@pytest.mark.parametrize("K", [8, 16])
@pytest.mark.parametrize("sea,jet", [(None, False), ((64, 1), False), ((64, 2), False), ((60, 1), False),
                                     (None, True), ((64, 2), True)])
def test_small_batch_rows_are_the_general_paths(gpu, K, sea, jet):
    print(f"case: K {K}, sea {sea}, jet {jet}", flush=True)
    hull = M.ico_ellipsoid(1.1, 0.5, 0.4, 5)
    c = 64 * K
    descs = []
    for i, m in enumerate((1, 63, 64, 65, c - 1, c, c + 1, 2 * c, 2 * c + 65, 5000)):
        for variant in range(3):
            descs.append(H.BodyDesc(mesh=H.Mesh(_part(hull, m)), volume=0.2, surface=1.0, buoyant=variant != 1,
                                    hydro=not (variant == 2 and i % 3 == 0)))
    descs.append(H.BodyDesc(mesh=H.Mesh(_part(hull, 20000, shuffle=True)), volume=0.2, surface=1.0))
    n = len(descs)
    rng = np.random.default_rng(7)
    st = _states(rng, n)
    go = _ocean(sea, jet)
    batch = H.BodyBatch(descs, faces_per_lane=K)
    batch.set_opts(K, 0, 1)
    ref = batch.compute_host(go, st, np.full((n, 24), 0.375))
    assert len(set(ref[:, 21])) == 4, "outside, inside, crossing and not hydrodynamic bodies"
    batch.set_opts(K, 0, 0)
    for _ in range(3):   # the chunk counters are zero again after every step
        _same_bits(batch.compute_host(go, st, np.full((n, 24), 0.375)), ref, (K, sea, jet))


@pytest.mark.parametrize("K", [8, 16])
@pytest.mark.parametrize("jet", [False, True])
def test_small_aero_batch_rows_are_the_general_paths(gpu, K, jet):
    print(f"case: aero K {K}, jet {jet}", flush=True)
    hull = M.ico_ellipsoid(1.1, 0.5, 0.4, 4)
    c = 64 * K
    descs = [H.AeroDesc(mesh=H.Mesh(_part(hull, m)), approx_params=np.array([1.1, 0.5, 0.4]), approx_type=3,
                        aero=k != 3) for k, m in enumerate((1, 64, 65, 500, c, c + 1, 5000))]
    n = len(descs)
    st = _states(np.random.default_rng(8), n)
    atm = H.Atmosphere(1.2)
    atm.add_uniform_current((4.0, 1.0, 0.0))
    if jet:
        atm.add_jet((30.0, 30.0, 0.5), (0.6, 0.8, 0.0), 30.0, 2.0)
    small = H.AeroBatch(descs, faces_per_lane=K)
    # the same bodies many times over: too many chunks for the one-launch step
    reps = -(-1100 // small.info()[1])
    large = H.AeroBatch(descs * reps, faces_per_lane=K)
    ref = large.compute_host(atm, np.tile(st, (reps, 1)), np.full((n * reps, 24), 0.375))
    for _ in range(2):
        _same_bits(small.compute_host(atm, st, np.full((n, 24), 0.375)), ref[:n], (K, jet))


def test_small_batch_mask_and_tick(gpu):
    """Masked steps write the active rows only, and the tick driver's forces
    are the rows' sums (zero off the overlap), on both paths."""
    import torch
    hull = M.ico_ellipsoid(1.1, 0.5, 0.4, 4)
    n = 24
    batch = H.BodyBatch([H.BodyDesc(mesh=H.Mesh(_part(hull, 300 + 190 * i)), volume=0.2, surface=1.0,
                                    hydro=i != 5) for i in range(n)])
    rng = np.random.default_rng(9)
    go = _ocean((64, 1), False)
    dev = torch.device("cuda", 0)
    rows, applied = [], []
    for split in (1, 0):
        batch.set_opts(0, 0, split)
        drv = H.TickDriver(batch, 2)
        out = torch.full((n, 24), 0.25, dtype=torch.float64, device=dev)
        app = torch.full((n, 6), 9.0, dtype=torch.float64, device=dev)
        rng = np.random.default_rng(9)
        for k in range(4):
            st = torch.from_numpy(_states(rng, n)).to(dev)
            ov = torch.from_numpy((rng.random(n) < 0.6).astype(np.uint8)).to(dev)
            drv.step(go, st.data_ptr(), ov.data_ptr(), out.data_ptr(), app.data_ptr())
            torch.cuda.synchronize()
            rows.append(out.cpu().numpy())
            applied.append(app.cpu().numpy())
    for k in range(4):
        _same_bits(rows[4 + k], rows[k], k)
        assert np.array_equal(applied[4 + k], applied[k]), k


@pytest.mark.parametrize("m", [1, 63, 64, 65, 511, 512, 513, 1025, 20480])
@pytest.mark.parametrize("shuffle", [False, True])
def test_per_body_calls_at_chunk_edges(gpu, m, shuffle):
    print(f"case: {m} faces, shuffled {shuffle}", flush=True)
    tm = _part(M.ico_ellipsoid(1.1, 0.5, 0.4, 5), m, shuffle)
    gm, om = H.Mesh(tm), O.Mesh.from_tri(tm)
    grid = W.grid_reference(W.pm_components(8, 5.0, 64.0, seed=3), 64).astype(np.float32)
    go = H.Ocean()
    go.set_waves(grid, 64, 1, [64.0])
    oo = O.Ocean(wave_data=grid, wave_n=64, channels=1, lengths=[64.0])
    rng = np.random.default_rng(m)
    st = _states(rng, 4, depth=(-0.4, 0.4))
    g, r, x = np.zeros((4, 24)), np.zeros((4, 24)), np.zeros((4, 22))
    gs, rs, xs = np.zeros((4, 24)), np.zeros((4, 24)), np.zeros((4, 22))
    for i, s in enumerate(st):
        outs, sv = [np.zeros(3) for _ in range(6)], np.zeros(2)
        H.ComputeHydrodynamicForcesSurface(H.HydrodynamicsSettings(True, True), gm, go, s[:16], s[:16], s[16:19],
                                           s[19:22], *outs, sv)
        g[i, :18], g[i, 18:20] = np.concatenate(outs), sv
        r[i], x[i] = O.surface(64, 1, 1, om, oo, s[:16], s[:16], s[16:19], s[19:22], full=True)
        outs = [np.zeros(3) for _ in range(4)]
        H.ComputeHydrodynamicForcesSubmerged(gm, go, s[:16], s[:16], s[16:19], s[19:22], *outs)
        gs[i, 6:18] = np.concatenate(outs)
        rs[i], xs[i] = O.submerged(64, om, oo, s[:16], s[:16], s[16:19], s[19:22], full=True)
        rs[i, 20] = 60   # drag vectors written
    for got, ref, ext, names in ((g, r, x, ("Fb", "Tb", "Fdq", "Tdq", "Fdf", "Tdf")),
                                 (gs, rs, xs, ("Fdq", "Tdq", "Fdf", "Tdf"))):
        worst, _ = bound_ratio(got, ref, ext, names)
        assert max(worst.values()) <= 1.0, worst
    np.testing.assert_allclose(g[:, 18], r[:, 18], rtol=1e-6, atol=1e-12)
