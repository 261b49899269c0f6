"""The launch rule of the 2D sweeps on either side of its line (1835008 cells)
and in the marching shapes it makes of grids of any form (one round of tiles,
several, narrow and short ones), against a caller's marching shapes."""
import numpy as np
import pytest
import torch

from tests.fields import cons_field

pytestmark = pytest.mark.gpu

SHAPES = [(1792, 1024), (1793, 1024),       # (ny, nx) at the line
          (1400, 1403), (7, 300007), (300007, 7), (2001, 2003), (33, 70001), (40000, 70)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype,layout", [(torch.float64, 1), (torch.float32, 0)], ids=str)
def test_rule_matches_callers_march(shape, dtype, layout):
    from fluidity_amd import euler as E
    U = cons_field("riemann", shape, seed=1001)
    a = np.moveaxis(U, -1, 0) if layout == 1 else U
    a = torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype=dtype)
    out = []
    for tuning in (None, dict(x_block=128, x_rows=16, y_block=64, y_rows=32)):
        s = E.SplitSolver(E.Scheme(bc=(1, 2, 0)), layout=layout)
        if tuning:
            s.set_tuning(**tuning)
        u = a.clone()
        r = s.simulate(u, torch.empty_like(u), 0.5, 1.0 / max(shape), max_iters=3)
        out.append((u, r.run_time, r.max_wavespeed))
    assert torch.equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
