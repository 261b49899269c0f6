"""Batches of problems at the edges of their tiles: lines of 56-cell segments,
planes of cell-parallel tiles (62 or 64 columns, 8 or 6 rows), against the
oracle and against the marching tiles of a caller's tuning."""
import numpy as np
import pytest
import torch

from tests.fields import cons_field

pytestmark = pytest.mark.gpu

SHAPES = [(4,), (55,), (56,), (57,), (447,), (448,), (449,), (897,),
          (4, 4), (6, 62), (7, 63), (8, 64), (9, 65), (13, 125), (131, 5)]


def _problems(E, dtype, layout, numerics, bc, flux):
    out = []
    for i, shape in enumerate(SHAPES):
        U = cons_field("smooth", shape, seed=40 + i)
        a = np.moveaxis(U, -1, 0) if layout == 1 else U
        out.append({"U": torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype=dtype),
                    "scheme": E.Scheme(flux=flux, gamma=1.3 + 0.02 * i, bc=bc,
                                       numerics=numerics),
                    "cfl": 0.8, "dh": 1.0 / shape[-1]})
    return out


def _run(B, problems, layout, steps, tuning=None):
    b = B.Batch(problems, layout=layout)
    if tuning:
        b.set_tuning(**tuning)
    b.step(steps)
    res = b.finish()
    return [b.state(i).cpu().numpy() for i in range(len(problems))], res


@pytest.mark.parametrize("bc", [(0, 1, 0), (1, 0, 0), (2, 2, 0)], ids=str)
@pytest.mark.parametrize("layout,flux", [(0, 0), (1, 0), (1, 1)])
def test_tile_edges_bitwise(oracle, bc, layout, flux):
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    steps = 7
    got, res = _run(B, _problems(E, torch.float64, layout, 0, bc, flux), layout, steps)
    for i, shape in enumerate(SHAPES):
        s = oracle.scheme(gamma=1.3 + 0.02 * i, bc=bc, flux=flux)
        U = cons_field("smooth", shape, seed=40 + i)
        ref, t, it, _ = oracle.simulate(U, s, 0.8, 1.0 / shape[-1], max_iters=steps)
        a = np.ascontiguousarray(np.moveaxis(got[i], 0, -1) if layout == 1 else got[i])
        assert (res[i].iters, res[i].run_time) == (it, t), shape
        assert np.array_equal(a.view(np.uint64), ref.view(np.uint64)), shape


@pytest.mark.parametrize("dtype,numerics", [(torch.float32, 0), (torch.float64, 1)], ids=str)
def test_tiles_match_marching_tiles(dtype, numerics):
    """The formulas round alike in every tile: FP32 bit for bit; the fast FP64
    maximum may leave out a cell within 5e-15 of it, and a step's dt with it
    (a state to about 1e-13 after the steps)."""
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    runs = [_run(B, _problems(E, dtype, 1, numerics, (0, 1, 0), 0), 1, 7, tuning)
            for tuning in (None, dict(x_block=64, x_rows=8, y_block=64, y_rows=16))]
    for a, b in zip(runs[0][0], runs[1][0]):
        if dtype == torch.float32:
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        else:
            assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
