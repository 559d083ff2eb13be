"""Steps that share a work buffer and are not ordered (two streams) leave their own
rows undefined and nothing else: once they have ended, every later step gives the
rows it gave before.  The no-alloc calls of one GPU share one buffer whatever
their meshes, a batch's steps share the batch's."""
import numpy as np
import pytest
import torch

from stonefish_amd import _native as N
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M

pytestmark = pytest.mark.gpu


def _state(z):
    s = np.zeros(38)
    s[[0, 5, 10, 15, 16, 21, 26, 31]] = 1.0
    s[14] = s[30] = z
    s[32:] = 0.4, -0.2, 0.1, 0.2, 0.1, -0.3
    return s


def test_noalloc_rows_after_overlapping_calls(gpu):
    print("case: no-alloc calls of four meshes after overlapping ones", flush=True)
    ocn, settings = H.Ocean(), H.HydrodynamicsSettings(True, True)
    meshes = [H.Mesh(M.ellipsoid_with_faces(1.0, 0.4, 0.3, f)) for f in (1500, 6000, 20000, 60000)]
    d_state = torch.from_numpy(_state(0.05)).cuda()

    def alone():
        rows = []
        for m in meshes:
            out = torch.full((24,), 7.0, dtype=torch.float64, device="cuda")
            H.forces_noalloc(settings, N.SFH_NOALLOC_SURFACE, m, ocn, d_state.data_ptr(), out.data_ptr())
            torch.cuda.synchronize()
            rows.append(out.cpu().numpy())
        return rows

    before = alone()
    assert all(np.abs(r[6:9]).max() > 0 and r[20] == 255 for r in before)
    streams = [torch.cuda.Stream() for _ in range(3)]
    sink = torch.zeros(3, 24, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for i in range(300):
        k = i % 3
        H.forces_noalloc(settings, N.SFH_NOALLOC_SURFACE, meshes[(i * 7 + k) % 4], ocn, d_state.data_ptr(),
                         sink[k].data_ptr(), streams[k].cuda_stream)
    torch.cuda.synchronize()
    for a, b in zip(before, alone()):
        assert np.array_equal(a, b)


def test_batch_rows_after_overlapping_steps(gpu):
    print("case: one-launch batch steps after overlapping ones", flush=True)
    ocn = H.Ocean()
    meshes = [H.Mesh(M.ellipsoid_with_faces(1.0, 0.4, 0.3, f)) for f in (900, 5000, 12000)]
    n = 60
    batch = H.BodyBatch([H.BodyDesc(mesh=meshes[i % 3], volume=0.5, surface=3.0) for i in range(n)], faces_per_lane=16)
    assert batch.info()[1] <= 1024
    st = np.stack([np.concatenate([_state(-0.25 + 0.02 * i)[:16], _state(0)[32:]]) for i in range(n)])
    d_st = torch.from_numpy(st).cuda()

    def alone():
        out = torch.full((n, 24), 7.0, dtype=torch.float64, device="cuda")
        batch.compute(ocn, d_st.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    before = alone()
    assert (np.abs(before[:, 6:9]).max(axis=1) > 0).all()
    streams = [torch.cuda.Stream() for _ in range(3)]
    sink = torch.zeros(3, n, 24, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for i in range(150):
        batch.compute(ocn, d_st.data_ptr(), sink[i % 3].data_ptr(), streams[i % 3].cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(before, alone())
