"""Reinitialisation of level sets that are steep or jump at the interface: a
neighbour across it enters with a large negated distance, so the band runs many
tiles past the sources.  Fields, bands and sweep counts of the oracle exactly.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _phi(kind, shape):
    n = shape[-1]
    x = (np.arange(n) + 0.5) / n
    if len(shape) == 1:
        if kind == "jump":
            return np.where(x < 0.4, -0.6 - 0.05 * x, 0.7 + 0.02 * x)
        return 150.0 * (np.abs(x - 0.5) - 0.1)
    y = (np.arange(shape[0]) + 0.5)[:, None] / n
    if kind == "jump":  # across a slanted line, its height varying along it
        return np.where(x + 0.7 * y < 0.45, -0.35 - 0.2 * y, 0.3 + 0.3 * y)
    return 60.0 * (np.hypot(x - 0.5, y - 0.5 * shape[0] / n) - 0.1 * shape[0] / n)


@pytest.mark.parametrize("kind", ["jump", "steep"])
@pytest.mark.parametrize("shape", [(3000,), (60, 400), (130, 170)], ids=str)
@pytest.mark.parametrize("band", [1, 6])
def test_reinit_band_past_the_sources(oracle, kind, shape, band):
    from fluidity_amd import levelset as L
    phi = np.broadcast_to(_phi(kind, shape), shape).copy()
    dh = 1.0 / shape[-1]
    ref, mask, its = oracle.ls_reinit(phi, dh, band)
    assert mask.sum() > 0
    got, bm, n = L.eikonal(torch.from_numpy(phi).to("cuda"), dh, band)
    assert n == its
    assert np.array_equal(bm.cpu().numpy(), mask)
    assert np.array_equal(got.cpu().numpy().view(np.uint64), ref.view(np.uint64))
