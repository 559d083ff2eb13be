"""A body's row does not depend on how many bodies are beside it.  On one wave
layer a batch of more than 12,288 chunks takes a crossing chunk's rows twice, from
records of its faces; a smaller one takes them once, from the vertices.  The
records hold what the vertices give, so all slots of the rows, the submerged
volume among them, are the same bits.  So are those of a masked step of the large
batch, which takes the rows once.  Hulls of fine and of coarse faces and a
revolved one with slivers at its pole, at every number of faces per lane that has
both ways."""
import numpy as np
import pytest
import torch

from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import transforms as T
from stonefish_amd import waves as W
from test_gpu_slivers import _sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 16, 32])
@pytest.mark.parametrize("layers", [1, 2])
def test_rows_do_not_depend_on_the_batch(gpu, K, layers):
    print(f"case: K {K}, {layers} layers", flush=True)
    n = 64
    data = np.zeros((n, n, layers), np.float32)
    for l in range(layers):
        data[:, :, l] = W.grid_reference(W.pm_components(8, 4.0, 64.0, seed=3 + l), n)
    go = H.Ocean()
    go.set_waves(data, n, layers, [64.0, 37.0][:layers])
    tris = [M.ico_ellipsoid(1.1, 0.5, 0.4, 4), M.ellipsoid_with_faces(0.9, 0.3, 0.25, 3001), M.box(0.9, 0.7, 0.3, 1),
            M.ico_ellipsoid(1.9, 1.3, 1.7, 1), _sphere(0.15, 32, 24)]
    meshes = [H.Mesh(t) for t in tris]
    few, many = 240, 13000
    descs = [H.BodyDesc(mesh=meshes[i % len(meshes)], volume=0.2, surface=1.0) for i in range(many)]
    rng = np.random.default_rng(7)
    st = np.zeros((many, 22))
    pos = np.stack([rng.uniform(0, 60, many), rng.uniform(0, 60, many), rng.uniform(-0.3, 0.3, many)], axis=1)
    st[:, :16] = T.quat_to_gl(T.random_unit_quaternions(rng, many), pos)
    st[:, 16:] = rng.uniform(-1, 1, (many, 6))
    small = H.BodyBatch(descs[:few], faces_per_lane=K, split_passes=1)
    large = H.BodyBatch(descs, faces_per_lane=K, split_passes=1)
    assert small.info()[1] <= 12288 < large.info()[1]
    a, b = small.compute_host(go, st[:few]), large.compute_host(go, st)[:few]
    assert (a[:, 21] == 2).sum() > few // 2 and (a[:, 19] > 0).sum() > few // 2
    for name, sl in {**H.OUT_FIELDS, "position": 21}.items():
        assert np.array_equal(a[:, sl], b[:, sl]), (name, np.abs(a[:, sl] - b[:, sl]).max())
    d_st = torch.from_numpy(st).cuda()
    mask = torch.zeros(many, dtype=torch.uint8, device="cuda")
    mask[:few:2] = 1
    out = torch.full((many, 24), 0.375, dtype=torch.float64, device="cuda")
    large.compute_masked(go, d_st.data_ptr(), mask.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    out = out.cpu().numpy()
    written = b[::2, :20] != 0.0   # slots the step leaves untouched keep the fill there, zero in b
    assert np.array_equal(out[:few:2, :20][written], b[::2, :20][written])
    assert np.array_equal(out[:few:2, 20:22], b[::2, 20:22]) and (out[1:few:2] == 0.375).all()
