"""The marching tiles of a batch (persistent workgroups that take tiles from a
counter, lines eight segments in turn) in the exact FP64 numerics against the
oracle, bit for bit, in both layouts (16-byte and single loads)."""
import numpy as np
import pytest
import torch

from tests.fields import cons_field
from tests.test_gpu_batch_tiles import SHAPES, _problems, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tuning", [dict(x_block=64, x_rows=8, y_block=64, y_rows=16),
                                    dict(x_block=256, x_rows=32, y_block=128, y_rows=5),
                                    dict(x_block=128, x_rows=4, y_block=64, y_rows=-16)], ids=str)
@pytest.mark.parametrize("layout,flux,bc", [(0, 0, (0, 1, 0)), (1, 0, (2, 2, 0)), (0, 1, (1, 0, 0)),
                                            (1, 1, (0, 2, 0))])
def test_marching_tiles_bitwise(oracle, tuning, layout, flux, bc):
    from fluidity_amd import euler as E
    from fluidity_amd import batch as B
    steps = 7
    got, res = _run(B, _problems(E, torch.float64, layout, 0, bc, flux), layout, steps, tuning)
    for i, shape in enumerate(SHAPES):
        s = oracle.scheme(gamma=1.3 + 0.02 * i, bc=bc, flux=flux)
        U = cons_field("smooth", shape, seed=40 + i)
        ref, t, it, _ = oracle.simulate(U, s, 0.8, 1.0 / shape[-1], max_iters=steps)
        a = np.ascontiguousarray(np.moveaxis(got[i], 0, -1) if layout == 1 else got[i])
        assert (res[i].iters, res[i].run_time) == (it, t), shape
        assert np.array_equal(a.view(np.uint64), ref.view(np.uint64)), shape
