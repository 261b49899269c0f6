"""One step's vector-Jacobian product where the adjoint's segments of 58 cells
begin and end, and on short lines, against the tape in plain PyTorch; the
tolerance is that of the step tests (rounding of reordered FP64 sums)."""
import numpy as np
import pytest
import torch

from tests.test_gpu_adjoint import A, E, _dev, _generic_state, _scheme, _soa, _tape_vjp  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [0, 1, 2])
@pytest.mark.parametrize("shape", [(58,), (59,), (60,), (61,), (117,), (7, 58), (5, 60), (58, 8),
                                   (59, 6), (61, 9), (117, 5)], ids=str)
def test_segment_edges(A, E, shape, bc):  # noqa: F811
    nd = len(shape)
    if nd == 1:
        U = _generic_state(1, nx=shape[0])
    else:
        side = max(shape)
        U = np.ascontiguousarray(_generic_state(2, ny=side, nx=side)[:shape[0], :shape[1]])
    bcs = (bc, (bc + 1) % 3)[:nd]
    flux, form = (("hllc", "cons"), ("force", "prim"), ("force", "cons"))[(sum(shape) + bc) % 3]
    lam = np.random.default_rng(sum(shape)).standard_normal(_soa(U).shape)
    dh = 1.0 / shape[-1]
    adj = A.Adjoint(_scheme(E, bcs, flux, form), 0.9, dh)
    got, dg = adj.step_vjp(_dev(U), torch.from_numpy(lam).to("cuda"))
    ref, dg_ref = _tape_vjp(U, lam, nd, bcs, 0.9, dh, flux=flux, form=form)
    scale = np.abs(ref).max()
    assert np.abs(got.cpu().numpy() - ref).max() <= 1e-11 * scale
    assert abs(dg - dg_ref) <= 1e-11 * max(abs(dg_ref), scale)
