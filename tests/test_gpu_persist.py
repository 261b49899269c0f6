"""The whole step loop of a 1D line in one launch against launched steps, at the
edges of its segments (56 cells a wave), workgroups (8 and 4 waves) and range.
"""
import numpy as np
import pytest
import torch

from tests.fields import cons_field

pytestmark = pytest.mark.gpu

CASES = [
    # cells, numerics or dtype, limiter, form, flux, boundary, layout, steps
    (4, "exact", 0, 0, 0, 0, 0, 7),
    (7, "exact", 0, 0, 0, 2, 1, 9),            # one segment, periodic
    (56, "fast", 0, 0, 0, 1, 0, 12),
    (57, "exact", 1, 1, 1, 1, 1, 12),          # two segments of 28 and 29 cells
    (448, "exact", 0, 0, 0, 2, 0, 21),         # one workgroup of 8 waves, periodic
    (449, "exact", 0, 1, 3, 2, 1, 21),         # three workgroups, periodic
    (1345, "f32", 0, 0, 0, 1, 0, 25),
    (5000, "fast", 1, 0, 2, 0, 1, 25),
    (57345, "exact", 0, 0, 1, 0, 0, 6),        # five waves a workgroup
    (229376, "f32", 1, 0, 0, 2, 1, 5),         # the last line of the range
    (229377, "fast", 0, 0, 0, 0, 1, 5),        # and the first past it
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:2])))
def test_loop_equals_launched_steps(case):
    from fluidity_amd import euler as E
    n, kind, lim, form, flux, bc, layout, steps = case
    U = cons_field("smooth", (n,), seed=n)
    dtype = torch.float32 if kind == "f32" else torch.float64
    out = []
    for graphs in (True, False):
        solver = E.SplitSolver(E.Scheme(limiter=lim, form=form, flux=flux, bc=(bc, 0, 0),
                                        numerics=1 if kind == "fast" else 0), layout=layout)
        solver.set_graphs(graphs)
        a = np.ascontiguousarray(np.moveaxis(U, -1, 0)) if layout == 1 else U
        a = torch.from_numpy(a).to("cuda", dtype=dtype)
        r = solver.simulate(a, torch.empty_like(a), 0.9, 1.0 / n, max_iters=steps)
        out.append((a.cpu(), r.iters, r.run_time, r.last_dt, r.max_wavespeed))
    assert torch.equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
    assert out[0][1] == steps
