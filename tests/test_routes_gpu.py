"""Which kernels the 2-D calls run on (MI355X): workgroup tiles, or the
wavefront tiles and in-place kernels where those measured faster, and the
latter against the CPU oracle over the forms of call that reach them.

Tolerances as in test_tiles_gpu.py: everything bit-identical but the FP64
coefficient gradients, which are reordered sums.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tide
from gpu_abi import gpu_backward, gpu_forward
from helpers import FIELD_NAMES, relative_l2
from oracle import oracle as O
from test_tiles_gpu import _case
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


def _families(fn):
    """Kernel families of the forward and of the adjoint that fn() runs."""
    for p in (0, 1):
        tide._native.take_tm2d_launches(p)
    fn()
    return [{k for k, n in enumerate(tide._native.take_tm2d_launches(p)) if n} for p in (0, 1)]


@pytest.mark.parametrize("case,forward,storing,adjoint", [
    (dict(ny=96, nx=96, shots=1, nt=64), TILES, TILES, TILES),
    (dict(ny=1065, nx=1065, shots=4, nt=64), TILES, TILES, TILES),
    (dict(ny=1300, nx=1300, shots=4, nt=64), TILES, TILES, WAVEFRONT),
    (dict(ny=1300, nx=1300, shots=4, nt=64, compression=True), TILES, TILES, TILES),
    (dict(ny=1300, nx=1300, shots=4, nt=24), TILES, TILES, TILES),
    (dict(ny=1300, nx=1300, shots=3, nt=64), TILES, TILES, TILES),
    (dict(ny=768, nx=800, shots=12, nt=64), TILES, WAVEFRONT, TILES),
    (dict(ny=441, nx=942, shots=12, nt=64), TILES, WAVEFRONT, TILES),
    (dict(ny=441, nx=942, shots=12, nt=64, compression=True), TILES, TILES, TILES),
    (dict(ny=700, nx=700, shots=4, nt=64, dtype=torch.float64), TILES, TILES, TILES),
    (dict(ny=96, nx=96, shots=2, nt=7, stencil=4), IN_PLACE, IN_PLACE, TILES),
    (dict(ny=96, nx=96, shots=2, nt=3, stencil=6), IN_PLACE, IN_PLACE, IN_PLACE),
    (dict(ny=96, nx=96, shots=2, nt=8, stencil=8), TILES, TILES, TILES),
    (dict(ny=420, nx=440, shots=4, nt=16, stencil=8, dtype=torch.float64), IN_PLACE,
     IN_PLACE, TILES),
    (dict(ny=400, nx=400, shots=4, nt=16, stencil=6, dtype=torch.float64), TILES, TILES, TILES),
    (dict(ny=110, nx=120, shots=40, nt=8, stencil=6, dtype=torch.float64), IN_PLACE,
     IN_PLACE, TILES),
    (dict(ny=64, nx=200, shots=40, nt=8, stencil=6, dtype=torch.float64), TILES, TILES, TILES),
    (dict(ny=64, nx=200, shots=40, nt=8, stencil=8, dtype=torch.float64), TILES, TILES, TILES),
])
def test_calls_run_on_the_kernels_that_measured_faster(case, forward, storing, adjoint):
    print(case, flush=True)
    case = dict(dict(stencil=2, dtype=torch.float32), **case)
    op, model, observed = _operator(**case)
    assert _families(lambda: op(model)) == [{forward}, set()]
    objective = ReceiverObjective(observed)
    assert (_families(lambda: objective.value_and_gradient(op.linearize(model)))
            == [{storing}, {adjoint}])


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
        assert _families(lambda: lin.jvp(direction)) == [{family}, set()]


@pytest.mark.parametrize("store,interval,batched,one", [
    ("full", 1, False, False), ("full", 1, True, False), ("full", 3, False, False),
    ("bf16", 1, False, False), ("bf16", 2, False, False), ("full", 1, False, True)])
@pytest.mark.parametrize("ny,nx,shots", [(41, 67, 7), (60, 75, 4)])
def test_wavefront_tiles_match_the_oracle(store, interval, batched, one, ny, nx, shots):
    """The two- and three-step wavefront tiles at their default shapes."""
    case = _case(ny, nx, 23, shots=shots, batched=batched)
    before = tide._native.get_tm2d_time_block()
    tide._native.set_tm2d_time_block(2, 3)
    try:
        for p in (0, 1):
            tide._native.take_tm2d_launches(p)
        f_o, r_o, es, cs = O.tm2d_forward(case, store=store, interval=interval)
        f_g, r_g, es_g, cs_g = gpu_forward(case, store=store, interval=interval)
        assert np.array_equal(r_g, r_o)
        assert np.array_equal(es_g, es) and np.array_equal(cs_g, cs)
        for name, a, b in zip(FIELD_NAMES, f_g, f_o):
            assert np.array_equal(a, b), name
        w = np.random.default_rng(3).standard_normal(r_o.shape).astype(case.dtype)
        ga_o, gb_o, gf_o, lam_o = O.tm2d_backward(case, w, es, cs, store=store, interval=interval)
        ga, gb, gf, lam = gpu_backward(case, w, es_g, None if one else cs_g, store=store,
                                       interval=interval)
        assert all(np.array_equal(a.reshape(b.shape), b) for a, b in zip(lam, lam_o))
        assert np.array_equal(gf, gf_o) and relative_l2(ga, ga_o) < 1e-12
        assert one or relative_l2(gb, gb_o) < 1e-12
        assert [tide._native.take_tm2d_launches(p)[WAVEFRONT] for p in (0, 1)] == [12, 8]
    finally:
        tide._native.set_tm2d_time_block(*before)


def test_the_kernel_timer_counts_the_launches_made():
    from tide.maxwell.tm2d import KernelTimer, set_kernel_timer

    op, model, observed = _operator(ny=96, nx=96, shots=2, nt=64, stencil=2, dtype=torch.float32)
    before = tide._native.get_tm2d_time_block()
    try:
        for block, family, launches in ((0, "tiles", (8, 8)), (2, "wavefront", (32, 32)),
                                        (3, "wavefront", (22, 22))):
            tide._native.set_tm2d_time_block(block, block)
            timer = KernelTimer()
            set_kernel_timer(timer)
            ReceiverObjective(observed).value_and_gradient(op.linearize(model))
            torch.cuda.synchronize()
            summary = timer.summary()
            for name, n in zip(("forward_store", "adjoint"), launches):
                assert summary[name]["launches"] == n and summary[name]["steps"] == 64
                assert summary[name]["steps_per_launch"] == round(64 / n)
                assert summary[name]["family"] == family
    finally:
        set_kernel_timer(None)
        tide._native.set_tm2d_time_block(*before)
