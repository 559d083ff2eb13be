"""The wave producer at the ends of its size range and an ocean whose field is
replaced: same size, another size, another number of layers, flat."""
import numpy as np
import pytest

import waves_fft as WF
from stonefish_amd import hydro as H
from stonefish_amd import meshes as M
from stonefish_amd import surrogate as S
from stonefish_amd import waves as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("passes", [1, 2, 6, 11])
def test_wave_producer_at_the_ends_of_its_range(gpu, passes):
    """A random spectrum against the FP64 oracle, with the bound of
    test_gpu_waves_fft.py: FP32 rounding through 2 P butterflies."""
    import torch
    n = 1 << passes
    rng = np.random.default_rng(passes)
    s12 = rng.normal(size=(n, n, 4)).astype(np.float32) * 0.05
    s34 = rng.normal(size=(n, n, 4)).astype(np.float32) * 0.01
    prod = W.WaveProducer(s12, s34, passes)
    out = torch.zeros((n, n, 4), dtype=torch.float32, device="cuda:0")
    prod.step(9.25, out.data_ptr())
    torch.cuda.synchronize()
    g = out.cpu().numpy().astype(np.float64)
    ref, Z = WF.heights(s12, s34, passes, W.REFERENCE_GRID_SIZES, 9.25)
    for c in range(4):
        bound = (8 * passes + 4) * 2.0 ** -24 * np.abs(Z[..., c // 2]).sum()
        assert np.abs(g[..., c] - ref[..., c]).max() <= bound, c
    prod.close()


def test_replaced_wave_field_is_the_new_one(gpu):
    hull = M.ico_ellipsoid(1.0, 0.5, 0.4, 3)
    n = 40
    batch = H.BodyBatch([H.BodyDesc(mesh=H.Mesh(hull), volume=0.8, surface=5.0)] * n)
    st = S.sample_states(np.random.default_rng(4), n, xy_range=(0.0, 60.0), depth_range=(-0.5, 1.0))
    rng = np.random.default_rng(5)
    ocean = H.Ocean()
    for size, channels, layers in ((64, 4, 2), (64, 4, 2), (64, 2, 2), (64, 1, 1), (60, 3, 1), (64, 4, 4), (0, 0, 0),
                                   (64, 4, 2)):
        fresh = H.Ocean()
        if size:
            data = (0.1 * rng.normal(size=(size, size, channels))).astype(np.float32)
            lengths = rng.uniform(30.0, 90.0, layers)
            for o in (ocean, fresh):
                o.set_waves(data, size, channels, lengths)
        else:
            ocean.set_waves(None, 0, 0, [])
        a, b = batch.compute_host(ocean, st), batch.compute_host(fresh, st)
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), (size, channels, layers)
        fresh.close()
