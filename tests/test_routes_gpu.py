"""Which kernels the 2-D calls run on (MI355X): workgroup tiles, or the
in-place kernels where those measured faster."""

from __future__ import annotations

import pytest
import torch

import tide
from tide.workflow import ReceiverObjective

pytestmark = pytest.mark.gpu

TILES, WAVEFRONT, IN_PLACE = range(3)


def _operator(ny, nx, shots, nt, stencil, dtype, compression=False, pml=8):
    """An operator on a padded ny x nx grid."""
    my, mx = (n - 2 * pml - stencil + 1 for n in (ny, nx))
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(3)
    eps = 1 + 8 * torch.rand(my, mx, generator=g, device=dev, dtype=dtype)
    dx = 0.01
    dt = 0.6 * dx / (2**0.5 * tide.C0)
    src = torch.tensor([[[1, (3 + 5 * s) % mx]] for s in range(shots)], device=dev)
    rec = torch.tensor([[[1, x] for x in range(0, mx, max(1, mx // 8))]] * shots, device=dev)
    amp = tide.ricker(6e8, nt, dt, dtype=dtype).reshape(1, 1, -1).repeat(shots, 1, 1).to(dev)
    op = tide.MaxwellTM(
        tide.Discretization(spacing=dx, dt=dt, stencil=stencil, boundary=tide.CPML(pml)),
        tide.Experiment(tide.Acquisition(src, rec), amp),
        storage=tide.StorageOptions(compression="bf16" if compression else False))
    model = tide.EMModel(eps, torch.zeros_like(eps), torch.ones_like(eps))
    return op, model, torch.zeros(nt, shots, rec.shape[1], device=dev, dtype=dtype)


def _family(fn):
    tide._native.take_tm2d_launches()
    fn()
    counts = tide._native.take_tm2d_launches()
    return {k for k, n in enumerate(counts) if n}


@pytest.mark.parametrize("case,forward,gradient", [
    # forward alone; forward with snapshots and adjoint of one gradient
    (dict(ny=96, nx=96, shots=1, nt=64), {TILES}, {TILES}),
    (dict(ny=1065, nx=1065, shots=4, nt=64), {TILES}, {TILES}),
    (dict(ny=1065, nx=1065, shots=4, nt=64, compression=True), {TILES}, {TILES}),
    (dict(ny=1065, nx=1065, shots=4, nt=24), {TILES}, {TILES}),
    (dict(ny=1065, nx=1065, shots=3, nt=64), {TILES}, {TILES}),
    (dict(ny=768, nx=800, shots=12, nt=64), {TILES}, {TILES}),
    (dict(ny=441, nx=942, shots=12, nt=64), {TILES}, {TILES}),
    (dict(ny=441, nx=942, shots=12, nt=64, compression=True), {TILES}, {TILES}),
    (dict(ny=700, nx=700, shots=4, nt=64, dtype=torch.float64), {TILES}, {TILES}),
    (dict(ny=96, nx=96, shots=2, nt=7, stencil=4), {IN_PLACE}, {IN_PLACE, TILES}),
    (dict(ny=96, nx=96, shots=2, nt=3, stencil=6), {IN_PLACE}, {IN_PLACE}),
    (dict(ny=96, nx=96, shots=2, nt=8, stencil=8), {TILES}, {TILES}),
    (dict(ny=400, nx=400, shots=4, nt=16, stencil=8, dtype=torch.float64), {IN_PLACE},
     {IN_PLACE, TILES}),
    (dict(ny=400, nx=400, shots=4, nt=16, stencil=6, dtype=torch.float64), {TILES}, {TILES}),
])
def test_calls_run_on_the_kernels_that_measured_faster(case, forward, gradient):
    print(case, flush=True)
    case = dict(dict(stencil=2, dtype=torch.float32), **case)
    op, model, observed = _operator(**case)
    assert _family(lambda: op(model)) == forward
    objective = ReceiverObjective(observed)
    assert _family(lambda: objective.value_and_gradient(op.linearize(model))) == gradient


@pytest.mark.parametrize("case,family", [
    (dict(ny=96, nx=96, shots=2, nt=2, stencil=2, dtype=torch.float32), TILES),
    (dict(ny=128, nx=128, shots=40, nt=8, stencil=8, dtype=torch.float64), IN_PLACE),
    (dict(ny=128, nx=128, shots=40, nt=8, stencil=8, dtype=torch.float32), TILES),
    (dict(ny=128, nx=128, shots=40, nt=8, stencil=6, dtype=torch.float64), TILES),
    (dict(ny=128, nx=128, shots=64, nt=8, stencil=6, dtype=torch.float64), IN_PLACE),
])
def test_jacobian_products_run_on_the_kernels_that_measured_faster(case, family):
    print(case, flush=True)
    op, model, _ = _operator(**case)
    direction = tide.EMDirection(epsilon=torch.ones_like(model.epsilon),
                                 sigma=torch.zeros_like(model.sigma))
    with op.linearize(model) as lin:
        assert _family(lambda: lin.jvp(direction)) == {family}
