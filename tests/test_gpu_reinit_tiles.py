"""Reinitialisation at the edges of its tiles (32 x 16 cells, 512 of a line)
and of its launches (four sweeps each): fields, bands and sweep counts of the
oracle exactly."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4,), (511,), (513,), (1030,), (15, 31), (16, 32), (17, 33),
                                   (5, 97), (65, 4), (50, 70)], ids=str)
@pytest.mark.parametrize("band", [1, 3, 6, 15])
def test_reinit_tile_edges(oracle, shape, band):
    from fluidity_amd import levelset as L
    rng = np.random.default_rng(17 + sum(shape) + band)
    n = shape[-1]
    x = [(np.arange(m) + 0.5) / n for m in shape]
    r = np.abs(x[0] - x[0].mean()) if len(shape) == 1 else np.hypot(
        x[0][:, None] - x[0].mean(), x[1][None, :] - 0.4)
    phi = 1.4 * (r - 0.6 * r.max()) + 0.002 * rng.normal(size=shape)
    out, mask, its = L.eikonal(torch.from_numpy(phi).to("cuda"), 1.0 / n, band)
    ref = oracle.ls_reinit(phi, 1.0 / n, band)
    assert its == ref[2]
    assert np.array_equal(mask.cpu().numpy(), ref[1])
    assert np.array_equal(out.cpu().numpy().view(np.uint64), ref[0].view(np.uint64))
