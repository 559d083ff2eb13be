"""The surrogate network's kernels at the edges of their tiles: inference in
tiles of 32 and of 64 rows, and the one-launch surrogate step in tiles of 32 and
of 64 units, give the same values."""
import numpy as np
import pytest

import mlp_ref as R

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _net(max_batch=256, seed=11):
    from stonefish_amd import surrogate as S
    net = S.Net(max_batch, 0)
    Ws, bs = R.init_weights(seed)
    for l in range(5):
        net.set_layer(l, Ws[l].numpy(), bs[l].numpy())
    return net, Ws, bs


@pytest.mark.parametrize("rows", [32, 64, 96, 24576, 24640, 24608, 40000])
def test_forward_is_independent_of_the_tile(gpu, rows):
    """The rows of one call against the same rows 32 at a time (always tiles of
    32): the sums run in the same order, so the bits agree."""
    net, _, _ = _net()
    x, _ = R.random_inputs(rows, rows)
    x = x.to(torch.bfloat16).cuda()
    y = torch.full((rows, 6), 7.0, device="cuda")
    net.forward(x, y)
    ref = torch.full((rows, 6), 9.0, device="cuda")
    for i in list(range(0, rows, 4096)) + [rows - 32]:
        j = min(rows, i + (32 if i == rows - 32 else 4096))
        net.forward(x[i:j], ref[i:j])
    torch.cuda.synchronize()
    assert torch.equal(y, ref)
    net.close()


def test_surrogate_step_is_independent_of_the_tile(gpu):
    """40 units by themselves (tiles of 32) and as the first of 8,300 (tiles of
    64, the last of a group partly filled).  The lanes that share a unit's wave
    queries are twice as many in the shorter tile, so its FP64 sums may differ
    in their last bits, far below the BF16 input of the network."""
    from stonefish_amd import hydro as H
    from stonefish_amd import meshes as M
    from stonefish_amd import surrogate as S
    from stonefish_amd import waves as W
    net, _, _ = _net()
    norm = S.Norm(np.zeros(13, np.float32), np.ones(13, np.float32), np.full(13, -3.0, np.float32),
                  np.full(13, 3.0, np.float32), np.zeros(6, np.float32), np.full(6, 0.2, np.float32))
    grid = W.grid_reference(W.pm_components(8, 5.0, 64.0, seed=3), 64).astype(np.float32)
    go = H.Ocean()
    go.set_waves(grid, 64, 1, [64.0])
    mesh = H.Mesh(M.ico_ellipsoid(1.0, 0.5, 0.4, 2))
    d = H.BodyDesc(mesh=mesh, volume=0.8, surface=5.0)
    n = 8300
    st = torch.from_numpy(S.sample_states(np.random.default_rng(2), n, xy_range=(0.0, 60.0))).cuda()
    got = []
    for m, counts in ((40, [40]), (n, [40, n - 40])):
        batch = H.BodyBatch([d] * m)
        step = S.SurrogateStep(batch, go, [net] * len(counts), [norm] * len(counts), counts, st[:m].contiguous())
        step.run()
        torch.cuda.synchronize()
        got.append((step.ft[:40].cpu(), step.ood[:40].cpu(), step.pos[:40].cpu()))
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2])
    assert set(got[0][2].tolist()) >= {1, 2}   # units inside and crossing
    err = (got[0][0] - got[1][0]).abs().max() / got[0][0].abs().max()
    assert float(err) < 1e-9, float(err)
    net.close()


@pytest.mark.parametrize("batch", [256, 768, 1280, 8192])
def test_gradients_at_batch_edges(gpu, batch):
    """One workgroup's rows, batches whose splits are fewer than the most, and
    a batch smaller than the one before it on the same network (whose
    transposed activations it must not see): the same bits as on a fresh
    network, and within the rounding of the FP32 reference."""
    x, t = R.random_inputs(90 + batch, batch)
    xd, td = x.to(torch.bfloat16).cuda(), t.cuda().contiguous()
    xl, tl = R.random_inputs(3, 9216)
    loss = torch.zeros(1, device="cuda")
    got = []
    for before in (False, True):
        net, Ws, bs = _net(9216, 21)
        if before:
            net.train_step(xl.to(torch.bfloat16).cuda(), tl.cuda().contiguous(), loss, lr=0.0)
        net.train_step(xd, td, loss, lr=0.0)
        got.append([g.cpu() for l in range(5) for g in net.gradients(l)] + [loss.cpu().clone()])
        net.close()
    for a, b in zip(*got):
        assert torch.equal(a, b)
    y, cache = R.forward(Ws, bs, x, rounded=True)
    lref, dy = R.loss_and_grad_out(y, t)
    dWs, dbs = R.backward(Ws, cache, dy, rounded=True)
    assert abs(float(got[0][10]) - float(lref)) <= 1e-3 * float(lref)
    for l in range(5):
        assert float((got[0][2 * l] - dWs[l]).norm() / dWs[l].norm()) < 1e-2, l
        assert float((got[0][2 * l + 1] - dbs[l]).norm() / dbs[l].norm()) < 1e-2, l
