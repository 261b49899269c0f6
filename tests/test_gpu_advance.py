"""The level-set stages of a two-material step (speeds, RK3, projection) on
ragged grids with rough level sets, and the one-sided derivatives that a wave
may leave out, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from fluidity_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(63, 33), (64, 32), (65, 31), (130, 61), (67, 64)])
def test_rough_level_sets_bitwise(oracle, nx, ny):
    from fluidity_amd import euler as E
    from fluidity_amd import levelset as L
    sb = W.shock_bubble(nx, ny, seed=1002)
    rng = np.random.default_rng(nx)
    phi = sb.phi0 + rng.uniform(-0.3, 0.3, size=sb.phi0.shape) * sb.dh
    sim = L.MultimaterialSimulator(layout=0)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
           for a in (sb.U0, sb.U1, phi, -phi)]
    for m, gamma in ((0, sb.gamma0), (1, sb.gamma1)):
        sim.add_material(dev[m], dev[2 + m], E.Scheme(gamma=gamma))
    r = sim.simulate_mm(0.5, sb.dh, max_iters=4, reinit_every=3)
    ref = oracle.mm_simulate(sb.U0, sb.U1, phi, -phi, oracle.scheme(gamma=sb.gamma0),
                             oracle.scheme(gamma=sb.gamma1), 0.5, sb.dh, max_iters=4,
                             reinit_every=3)
    assert (r.iters, r.run_time) == (ref[5], ref[4])
    for a, b in zip(dev, ref[:4]):
        assert np.array_equal(a.cpu().numpy().view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("bad", [None, np.nan, np.inf, 1e60, 1e200])
def test_advect_left_out_derivatives(oracle, bad):
    """Monotone regions (one derivative left out), kinks, constant patches,
    and single cells that are not finite or overflow the weights."""
    from fluidity_amd import levelset as L
    ny, nx = 48, 200
    y, x = np.mgrid[0:ny, 0:nx] * (1.0 / nx)
    phi = np.abs(x - 0.41) - 0.1 + 0.3 * np.abs(y - 0.1)
    phi[:, 150:] = phi[:, 150:150 + 1]
    phi[30:, 150:] = 0.7
    if bad is not None:
        for j, i in ((5, 20), (9, 100), (17, 170), (40, 190)):
            phi[j, i] = bad
    V = np.sin(40.0 * x) * np.cos(30.0 * y)
    V[:, 60:70] = 0.0
    dh, dt = 1.0 / nx, 0.3 / nx
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda") for a in (phi, V)]
    out = L.evolve(*dev, dt, dh).cpu().numpy()
    ref = oracle.ls_advect(phi, V, dt, dh)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(out[ok].view(np.uint64), ref[ok].view(np.uint64))
