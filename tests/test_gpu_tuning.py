"""A tuning that a context, a batch or the autotuner reports reproduces what
runs when it is set again, there or elsewhere."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.fields import cons_field

pytestmark = pytest.mark.gpu


def _tuple(t):
    return t.x_block, t.x_rows, t.y_block, t.y_rows


def _set(target, t):
    target.set_tuning(**dict(zip(("x_block", "x_rows", "y_block", "y_rows"), _tuple(t))))


def _grid(shape, seed=2):
    return torch.from_numpy(np.ascontiguousarray(np.moveaxis(cons_field("smooth", shape, seed), -1, 0))).cuda()


def test_context_tuning_round_trip():
    from fluidity_amd import euler as E
    from fluidity_amd import native as N
    s = E.SplitSolver(E.Scheme(), layout=1)
    fresh = s.ctx.get_tuning()
    assert fresh.x_rows == fresh.y_rows == N.FL_ROWS_RULE
    _set(s, fresh)
    assert _tuple(s.ctx.get_tuning()) == _tuple(fresh)
    s.set_tuning(x_block=128, x_rows=18)             # y keeps the rule
    t = s.ctx.get_tuning()
    assert _tuple(t)[:2] == (128, 18) and t.y_rows == N.FL_ROWS_RULE
    s.set_tuning()                                   # zeros change nothing
    assert _tuple(s.ctx.get_tuning()) == _tuple(t)
    s.set_tuning(x_rows=-16, y_block=64, y_rows=-43)
    assert _tuple(s.ctx.get_tuning()) == (128, -16, 64, -43)
    _set(s, fresh)
    assert s.ctx.get_tuning().x_rows == s.ctx.get_tuning().y_rows == N.FL_ROWS_RULE
    before = _tuple(s.ctx.get_tuning())
    for bad in (dict(x_rows=4097), dict(y_rows=-4097), dict(x_block=96, y_rows=8), dict(y_block=320)):
        with pytest.raises(N.FluidityError):
            s.set_tuning(**bad)
        assert _tuple(s.ctx.get_tuning()) == before


def test_autotuned_choice_carries_over():
    """On a small grid the cell-parallel sweeps are two to three times as fast
    as the best march: the autotuner picks them and says so."""
    from fluidity_amd import euler as E
    from fluidity_amd import native as N
    U = _grid((64, 64))
    a = E.SplitSolver(E.Scheme(), layout=1)
    t = a.autotune(U.clone(), torch.empty_like(U), reps=3)
    assert t.x_rows < 0 and t.y_rows < 0
    assert _tuple(t) == _tuple(a.ctx.get_tuning())
    b = E.SplitSolver(E.Scheme(), layout=1)
    _set(b, t)
    assert _tuple(b.ctx.get_tuning()) == _tuple(t)
    out = []
    for s in (a, b):
        u = U.clone()
        r = s.simulate(u, torch.empty_like(u), 0.8, 1.0 / 64, max_iters=6)
        out.append((u, r.run_time))
    u = U.clone()
    w = torch.empty_like(u)
    f, fw = E.grid_field(u, 1), E.grid_field(w, 1)
    p, r, sc = N.SimParams(0.8, 1.0 / 64, float("inf"), 6), N.SimResult(), E.Scheme().c()
    N.check(N.lib.fl_simulate_noalloc(C.byref(t), C.byref(f), C.byref(fw), C.byref(sc), C.byref(p),
                                      C.byref(r), torch.cuda.current_stream().cuda_stream))
    out.append((u, r.run_time))
    for u, rt in out[1:]:
        assert torch.equal(u, out[0][0]) and rt == out[0][1]


def test_batch_tuning_round_trip():
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    from fluidity_amd import native as N

    def batch():
        return B.Batch([{"U": _grid(s, 4), "scheme": E.Scheme(), "cfl": 0.8, "dh": 1.0 / s[-1]}
                        for s in ((40, 60), (33,), (64, 64))], layout=1)
    b = batch()
    fresh = b.get_tuning()
    assert fresh.x_rows < 0 and fresh.y_rows < 0     # small: cell-parallel tiles
    ref = None
    for t in (fresh, N.Tuning(64, 8, 64, 16), N.Tuning(64, -8, 64, 16),
              N.Tuning(64, N.FL_ROWS_RULE, 64, N.FL_ROWS_RULE)):
        c = batch()
        _set(c, t)
        got = c.get_tuning()
        want = [-abs(r) if r < 0 else r for r in (t.x_rows, t.y_rows)]
        assert [np.sign(got.x_rows), np.sign(got.y_rows)] == [np.sign(r) for r in want]
        if N.FL_ROWS_RULE not in want:
            assert _tuple(got) == _tuple(t)
        c.step(5)
        c.finish()
        states = [c.state(i) for i in range(3)]
        ref = ref or states
        assert all(torch.equal(x, y) for x, y in zip(states, ref))
    t = b.autotune(reps=2)
    assert _tuple(t) == _tuple(b.get_tuning())
    c = batch()
    _set(c, t)
    assert _tuple(c.get_tuning()) == _tuple(t)


def test_batch_zeros_keep_each_phase():
    """All zeros, or the values of one phase alone, leave the tiles of the
    phases they do not name as they are."""
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    b = B.Batch([{"U": _grid((40, 60)), "scheme": E.Scheme(), "cfl": 0.8, "dh": 1.0 / 60}], layout=1)
    fresh = _tuple(b.get_tuning())
    assert fresh[1] < 0 and fresh[3] < 0
    b.set_tuning()
    assert _tuple(b.get_tuning()) == fresh
    b.set_tuning(x_block=64, x_rows=8)
    assert _tuple(b.get_tuning()) == (64, 8) + fresh[2:]
    b.set_tuning(y_block=64, y_rows=16)
    assert _tuple(b.get_tuning()) == (64, 8, 64, 16)
    b.set_tuning()
    assert _tuple(b.get_tuning()) == (64, 8, 64, 16)


def _hip():
    for line in open("/proc/self/maps"):
        if "libamdhip64.so" in line:
            return C.CDLL(line.split()[-1])
    raise RuntimeError("no HIP runtime in this process")


def test_batch_survives_a_failed_autotune():
    """While a stream captures in global mode the uploads of the autotuner are
    refused: the call fails, and the steps after it are those of the tiles that
    the batch had, its 1D problems (here after an odd step count) included."""
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    from fluidity_amd import native as N

    def batch():
        return B.Batch([{"U": _grid(s, 4), "scheme": E.Scheme(), "cfl": 0.8, "dh": 1.0 / s[-1]}
                        for s in ((90, 130), (333,), (64, 64))], layout=1)
    hip = _hip()
    ref = batch()
    ref.step(7)
    for tuning in (None, dict(x_block=64, x_rows=8, y_block=64, y_rows=16)):
        b = batch()
        if tuning:
            b.set_tuning(**tuning)
        had = _tuple(b.get_tuning())
        b.step(3)
        torch.cuda.synchronize()
        stream, graph = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        with pytest.raises(N.FluidityError):
            b.autotune(reps=1)
        hip.hipStreamEndCapture(stream, C.byref(graph))
        if graph:
            hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)
        hip.hipGetLastError()
        assert _tuple(b.get_tuning()) == had
        b.step(4)
        got, want = b.finish(), ref.finish()
        for i in range(3):
            assert torch.equal(b.state(i), ref.state(i))
            assert (got[i].iters, got[i].run_time) == (want[i].iters, want[i].run_time) == (7, want[i].run_time)


def test_batch_of_many_fp32_cells_on_lines_marches():
    """The rule of the lines, and its marching tiles against the register tiles
    of a caller's tuning, bit for bit."""
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E
    shapes = [(65536 - 13 * i,) for i in range(56)] + [(40, 60)]
    assert 3 << 20 < sum(s[0] for s in shapes[:-1])

    def batch(dtype):
        r = np.random.default_rng(3)
        return B.Batch([{"U": (_grid(s, 4) * (1.0 + 0.01 * r.random())).to(dtype),
                         "scheme": E.Scheme(), "cfl": 0.8, "dh": 1.0 / s[-1]} for s in shapes], layout=1)
    b, c = batch(torch.float32), batch(torch.float32)
    assert b.get_tuning().x_rows > 0 and b.get_tuning().y_rows < 0
    c.set_tuning(x_rows=-32)
    for x in (b, c):
        x.step(3)
        x.finish()
    assert all(torch.equal(b.state(i), c.state(i)) for i in range(len(shapes)))
    assert batch(torch.float64).get_tuning().x_rows < 0


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=str)
def test_batch_autotune_inside_a_run(dtype):
    """The timed phases reduce into the slots that the next step clears and run
    state -> work: a run goes on as if there had been none, from odd and even
    step counts, problems that have stopped included."""
    from fluidity_amd import batch as B
    from fluidity_amd import euler as E

    def batch():
        return B.Batch([{"U": _grid(s, 4).to(dtype), "scheme": E.Scheme(), "cfl": 0.8,
                         "dh": 1.0 / s[-1], "max_iters": 5 if i == 1 else 100}
                        for i, s in enumerate(((90, 130), (333,), (64, 64), (2000,)))], layout=1)
    ref = batch()
    ref.step(13)
    want = ref.finish()
    b = batch()
    for steps in (4, 3, 6):
        b.step(steps)
        b.autotune(reps=1)
    got = b.finish()
    for i in range(4):
        assert torch.equal(b.state(i), ref.state(i))
        assert [got[i].iters, got[i].run_time, got[i].max_wavespeed] == \
            [want[i].iters, want[i].run_time, want[i].max_wavespeed]
