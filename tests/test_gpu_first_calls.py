"""The first step after an allocation counts on counters that were cleared just
before it: the per-body calls of a new or grown workspace, on their own
non-blocking stream, and the first one-launch step of a new batch on the
caller's.  They are made here while the null stream is busy, which a
non-blocking stream does not wait for, and give the rows of the same calls made
again on an idle GPU."""
import threading

import numpy as np
import pytest
import torch

from stonefish_amd import hydro as H
from stonefish_amd import meshes as M

pytestmark = pytest.mark.gpu


def _busy_null_stream():
    """Some tens of milliseconds of work on the null stream; the memory it frees
    holds ones in every bit."""
    torch.full((64 << 20,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    a = torch.randn(4096, 4096, device="cuda")
    b = a
    for _ in range(40):
        b = a @ b
        b = b / b.abs().max()
    return b


def _pose(z):
    t = np.eye(4)
    t[:3, 3] = 0.0, 0.0, z
    return t.T.reshape(-1).copy()


def test_first_per_body_calls_beside_a_busy_null_stream(gpu):
    print("case: first per-body calls of new and grown workspaces", flush=True)
    meshes = [H.Mesh(M.ellipsoid_with_faces(1.0, 0.4, 0.3, f)) for f in (700, 6000, 60000)]
    ocn = H.Ocean()
    eye, v, w = np.eye(4).reshape(-1).copy(), np.array([0.6, -0.2, 0.1]), np.array([0.1, 0.2, -0.3])

    def calls(i):
        rows = []
        for m in meshes:
            out = np.zeros((4, 3))
            H.ComputeHydrodynamicForcesSubmerged(m, ocn, _pose(5.0 + i), eye, v, w, *out)
            rows.append(out)
        return rows

    got = [None] * 8
    gate = threading.Barrier(8)

    def work(i):
        gate.wait()
        got[i] = calls(i)

    busy = _busy_null_stream()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert torch.isfinite(busy).all()
    for i in range(8):
        for a, b in zip(got[i], calls(i)):
            assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_first_batch_step_beside_a_busy_null_stream(gpu):
    print("case: first one-launch step of a new batch", flush=True)
    mesh = H.Mesh(M.ellipsoid_with_faces(1.0, 0.4, 0.3, 12000))
    ocn = H.Ocean()
    n = 40
    st = np.zeros((n, 22))
    for i in range(n):
        st[i, :16] = _pose(-0.2 + 0.05 * i)
    st[:, 16:] = 0.3
    d_st = torch.from_numpy(st).cuda()
    d_out, d_again = (torch.zeros(n, 24, dtype=torch.float64, device="cuda") for _ in range(2))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    busy = _busy_null_stream()
    batch = H.BodyBatch([H.BodyDesc(mesh=mesh, volume=0.5, surface=3.0)] * n, faces_per_lane=16)
    assert n < batch.info()[1] <= 1024
    batch.compute(ocn, d_st.data_ptr(), d_out.data_ptr(), s.cuda_stream)
    s.synchronize()
    torch.cuda.synchronize()
    assert torch.isfinite(busy).all()
    batch.compute(ocn, d_st.data_ptr(), d_again.data_ptr(), s.cuda_stream)
    s.synchronize()
    got, again = d_out.cpu().numpy(), d_again.cpu().numpy()
    assert (np.abs(again[:, 6:9]).max(axis=1) > 0).all() and np.array_equal(got, again)
