"""fl_simulate's captured steps against launching every kernel, bit for bit:
loops of 72 steps and more (captured at once: runs of 18 steps, the steps left
over, more than one batch of 252) and shorter ones from their second call on,
2D grids and lines beyond the persistent loop (three slots of the maximum), in
loops that a stop time ends, with other work between the replays."""
import numpy as np
import pytest
import torch

from tests.fields import cons_field

pytestmark = pytest.mark.gpu


def _run(E, U, graphs, calls, layout, dtype, **kw):
    """`calls` runs from the same state with one solver; the results of each."""
    a = np.moveaxis(U, -1, 0) if layout == 1 else U
    a = torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype=dtype)
    s = E.SplitSolver(E.Scheme(bc=(2, 1, 0)), layout=layout)
    s.set_graphs(graphs)
    u, w, other = torch.empty_like(a), torch.empty_like(a), torch.empty_like(a)
    out = []
    for _ in range(calls):
        u.copy_(a)
        s.sweep(a, other, 0, 0.01)                   # eager work of the same context
        s.max_wavespeed(other)
        torch.cuda.synchronize()
        r = s.simulate(u, w, 0.6, 1.0 / U.shape[-2], **kw)
        out.append((u.clone(), r.iters, r.run_time, r.last_dt, r.max_wavespeed))
    return out


def _same(E, U, calls, layout, dtype, **kw):
    ref = _run(E, U, False, 1, layout, dtype, **kw)[0]
    for got in _run(E, U, True, calls, layout, dtype, **kw):
        assert got[1:] == ref[1:]
        assert torch.equal(got[0], ref[0])
    return ref


@pytest.mark.parametrize("steps", [72, 85, 108, 253, 300])
@pytest.mark.parametrize("shape,layout,dtype", [((40, 52), 1, torch.float64), ((9, 130), 0, torch.float32)],
                         ids=str)
def test_long_loops(E, steps, shape, layout, dtype):
    ref = _same(E, cons_field("smooth", shape, 0), 3, layout, dtype, max_iters=steps)
    assert ref[1] == steps


@pytest.mark.parametrize("steps", [1, 13, 18, 19, 45])
@pytest.mark.parametrize("shape", [(40, 52), (70, 64)])
def test_short_loops_from_the_second_call(E, steps, shape):
    ref = _same(E, cons_field("smooth", shape, 0), 4, 1, torch.float64, max_iters=steps)
    assert ref[1] == steps


@pytest.mark.parametrize("steps", [73, 91])
@pytest.mark.parametrize("layout,dtype", [(1, torch.float64), (0, torch.float32)], ids=str)
def test_lines_beyond_the_persistent_loop(E, steps, layout, dtype):
    """Odd counts leave the result in the work buffer, which is copied back."""
    ref = _same(E, cons_field("smooth", (229400,), 0), 2, layout, dtype, max_iters=steps)
    assert ref[1] == steps


@pytest.mark.parametrize("shape", [(40, 52), (229400,)])
def test_stop_time_inside_a_run(E, shape):
    U = cons_field("smooth", shape, 0)
    full = _run(E, U, False, 1, 1, torch.float64, max_iters=90)[0]
    ref = _same(E, U, 2, 1, torch.float64, max_iters=90, sim_time=0.7 * full[2])
    assert 0 < ref[1] < 90


def test_other_parameters_between_the_calls(E):
    """A second loop with other parameters on the same solver, then the first again."""
    U = cons_field("smooth", (40, 52), 0)
    a = torch.from_numpy(np.ascontiguousarray(np.moveaxis(U, -1, 0))).cuda()
    out = []
    for graphs in (True, False):
        s = E.SplitSolver(E.Scheme(), layout=1)
        s.set_graphs(graphs)
        u, w = torch.empty_like(a), torch.empty_like(a)
        for cfl, steps in ((0.6, 20), (0.6, 20), (0.5, 80), (0.6, 20), (0.6, 20), (0.5, 80)):
            u.copy_(a)
            r = s.simulate(u, w, cfl, 1.0 / 52, max_iters=steps)
            out.append((graphs, u.clone(), r.iters, r.run_time, r.last_dt, r.max_wavespeed))
    half = len(out) // 2
    for g, e in zip(out[:half], out[half:]):
        assert torch.equal(g[1], e[1]) and g[2:] == e[2:]


@pytest.fixture(scope="module")
def E():
    from fluidity_amd import euler
    return euler
