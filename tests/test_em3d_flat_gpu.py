"""The 3-D step kernels, which take 256 (fp64: 128) consecutive cells of a
volume per wavefront, against the CPU oracle where that split can go wrong:
volumes that end inside a chunk or fill it, rows shorter than a vector's
reach and longer than a chunk, no CPML on a side, doubled sources, and more
receivers in a chunk than a wavefront has lanes.

Fields, receivers, snapshots, adjoint fields and source gradients are
bit-identical (the same expressions in their order); FP64 coefficient
gradients within 1e-12, the bound of a reordered sum over shots and steps.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_abi import gpu_em3d_backward, gpu_em3d_forward
from helpers import hetero3d_problem, relative_l2
from oracle import oracle as O
from tide.maxwell.maxwell3d import prepare_em3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape,pml,shots", [
    ((5, 5, 5), (1, 0, 1, 0, 1, 0), 1),
    ((6, 5, 5), (0, 0, 0, 0, 0, 0), 2),
    ((5, 6, 300), (2, 1, 1, 2, 12, 3), 2),
    ((9, 25, 22), (3, 3, 3, 3, 4, 4), 1),   # 16 x 32 x 31
    ((9, 25, 23), (3, 3, 3, 3, 4, 4), 3),   # 16 x 32 x 32: whole chunks
])
def test_chunks_of_a_volume_match_the_oracle(shape, pml, shots, dtype):
    nz, ny, nx = shape
    case = O.em_case_from_setup(prepare_em3d(**hetero3d_problem(
        dtype=dtype, nz=nz, ny=ny, nx=nx, nt=14, shots=shots, pml=pml, src_comp="ez",
        rec_comp="ex")))
    pz, py, px = case.shape
    print(f"case {case.shape} {dtype} shots {shots}", flush=True)
    rng = np.random.default_rng(2)

    def cells(n):
        z, y, x = (rng.integers(1, m, size=(shots, n)) for m in (pz, py, px))
        return (z * py + y) * px + x

    case.rec = cells(150)
    case.rec[:, 1] = case.rec[:, 0]
    case.src = np.repeat(cells(2), 2, axis=1)
    case.f = rng.standard_normal((case.nt, shots, 4)).astype(case.dtype)
    for store in ("full", "bf16") if dtype == torch.float32 else ("full",):
        f_o, r_o, s_o = O.em3d_forward(case, store=store)
        f_g, r_g, s_g = gpu_em3d_forward(case, store=store)
        assert np.abs(r_o).max() > 0 and np.array_equal(r_g, r_o)
        assert all(np.array_equal(a, b) for a, b in zip(f_g, f_o))
        assert all(np.array_equal(a, b) for a, b in zip(s_g, s_o))
        w = rng.standard_normal(r_o.shape).astype(case.dtype)
        gg = gpu_em3d_backward(case, w, s_o, store=store)
        go = O.em3d_backward(case, w, s_o, store=store)
        assert all(np.array_equal(a, b) for a, b in zip(gg[3], go[3]))
        assert np.array_equal(gg[2], go[2])
        assert relative_l2(gg[0], go[0]) < 1e-12 and relative_l2(gg[1], go[1]) < 1e-12
