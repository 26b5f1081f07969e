"""Workgroup tiles of the 2-D TM time loops (one launch advances a tile by
several steps) against the CPU oracle, at the edges of their shapes: grids
narrower than a tile, one column or row beside a tile's owned cells, every
remainder of the time loop, per-shot coefficients, several points in one
cell and points in several rows.

Tolerances: fields, receivers, snapshots, adjoint fields and source
gradients bit-identical (the single-step expressions in their order, and an
exactly rounded CPML division); FP64 coefficient gradients within 1e-12, the
bound of a reordered sum of nt * shots terms.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tide
from gpu_abi import gpu_backward, gpu_forward
from helpers import FIELD_NAMES, relative_l2
from oracle import oracle as O
from tide.maxwell.tm2d import prepare_tm2d

gpu = pytest.mark.gpu


def _case(ny, nx, nt, *, stencil=2, dtype=torch.float32, shots=2, pml=(3, 4, 5, 2), batched=False,
          seed=5):
    """A padded ny x nx problem with doubled points and two source rows."""
    half = stencil // 2
    my, mx = ny - pml[0] - pml[1] - 2 * half + 1, nx - pml[2] - pml[3] - 2 * half + 1
    g = torch.Generator().manual_seed(seed)
    shape = (shots, my, mx) if batched else (my, mx)
    eps = (1.0 + 8.0 * torch.rand(*shape, generator=g, dtype=torch.float64)).to(dtype)
    sig = (0.01 * torch.rand(*shape, generator=g, dtype=torch.float64)).to(dtype)
    dx = 0.01
    dt = 0.7 * dx / (2**0.5 * tide.C0)
    amp = tide.ricker(9e8, nt + 8, dt, peak_time=4 * dt, dtype=dtype)[:nt].reshape(1, 1, -1)
    amp = amp.repeat(shots, 3, 1) * torch.tensor([1.0, 0.5, -0.7], dtype=dtype)[None, :, None]
    src = torch.stack([torch.tensor([[1, (2 + 3 * s) % mx], [1, (2 + 3 * s) % mx], [my - 1, s % mx]])
                       for s in range(shots)])
    cols = list(range(0, mx, 2)) + [1 % mx, 1 % mx]
    rec = torch.stack([torch.tensor([[1, x] for x in cols] + [[my // 2, 0]])] * shots)
    st = prepare_tm2d(eps, sig, torch.ones_like(eps), dx, dt, amp, src, rec, stencil=stencil,
                      pml_width=list(pml))
    assert (st.ny, st.nx) == (ny, nx)
    return O.case_from_setup(st)


def _check(case, store="full"):
    f_o, r_o, es, cs = O.tm2d_forward(case, store=store)
    f_g, r_g, es_g, cs_g = gpu_forward(case, store=store)
    assert np.array_equal(r_g, r_o)
    assert np.array_equal(es_g, es) and np.array_equal(cs_g, cs)
    for name, a, b in zip(FIELD_NAMES, f_g, f_o):
        assert np.array_equal(a, b), name
    f_n, r_n, _, _ = gpu_forward(case)
    assert np.array_equal(r_n, r_o) and all(np.array_equal(a, b) for a, b in zip(f_n, f_o))
    w = np.random.default_rng(3).standard_normal(r_o.shape).astype(case.dtype)
    ga_o, gb_o, gf_o, lam_o = O.tm2d_backward(case, w, es, cs, store=store)
    ga, gb, gf, lam = gpu_backward(case, w, es_g, cs_g, store=store)
    for a, b in zip(lam, lam_o):
        assert np.array_equal(a.reshape(b.shape), b)
    assert np.array_equal(gf, gf_o)
    for a, b in ((ga, ga_o), (gb, gb_o)):  # a single step from rest has no gradient
        assert relative_l2(a, b) < 1e-12 if b.any() else not a.any()


@gpu
@pytest.mark.parametrize("ny,nx", [(14, 14), (48, 64), (49, 65), (47, 63), (17, 130), (97, 33),
                                   (128, 49)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_grids_beside_the_tile_edges(ny, nx, dtype):
    print(f"grid {ny}x{nx} {dtype}", flush=True)
    _check(_case(ny, nx, 21, dtype=dtype))


@gpu
@pytest.mark.parametrize("nt", [1, 2, 7, 8, 9, 15, 16, 17, 33])
def test_every_remainder_of_the_time_loop(nt):
    print(f"nt {nt}", flush=True)
    _check(_case(40, 70, nt))


@gpu
def test_many_tiles_and_shots_take_the_larger_tiles():
    _check(_case(230, 310, 13, shots=7, pml=(12, 9, 11, 10)))


@gpu
@pytest.mark.parametrize("stencil,ny,nx", [(4, 18, 18), (4, 46, 92), (4, 93, 47), (6, 35, 69),
                                           (8, 33, 51)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nt", [1, 10])
def test_higher_orders_beside_the_tile_edges(stencil, ny, nx, dtype, nt):
    print(f"order {stencil} grid {ny}x{nx} {dtype} nt {nt}", flush=True)
    _check(_case(ny, nx, nt, stencil=stencil, dtype=dtype))


@gpu
def test_bf16_snapshots_and_per_shot_coefficients():
    _check(_case(60, 75, 19, shots=3), store="bf16")
    _check(_case(60, 75, 19, shots=3, batched=True))


def test_cpml_division_by_held_reciprocal_is_exact():
    """d / k rounded to 32 bits equals the 64-bit product d * (1 / k)
    rounded to 32 bits: a quotient of two 24-bit numbers lies at least 2^-49
    (relative) from the midpoint of two floats, the product within 2^-52 of
    the quotient.  Random bit patterns (subnormals, infinities and NaN
    included) over the range of the CPML stretch."""
    rng = np.random.default_rng(1)
    d = rng.integers(0, 1 << 32, 4_000_000, dtype=np.uint64).astype(np.uint32).view(np.float32)
    k = rng.integers(0x3F800000, 0x40A00001, d.size, dtype=np.uint64).astype(np.uint32).view(np.float32)
    with np.errstate(all="ignore"):
        want = d / k
        got = (d.astype(np.float64) * (1.0 / k.astype(np.float64))).astype(np.float32)
    assert np.array_equal(got, want, equal_nan=True)
    assert np.array_equal(np.signbit(got[want == 0]), np.signbit(want[want == 0]))


def _born(case, dca, dcb, df):
    """born_forward on an oracle case (dca = dcb = None: no scattering)."""
    ptr = lambda t: 0 if t is None else tide._native.ptr(t)  # noqa: E731
    dtype = torch.from_numpy(case.ca).dtype
    d = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)  # noqa: E731
    bg, sc = [d(x) for x in case.fields], [d(np.zeros_like(x)) for x in case.fields]
    r = torch.zeros(case.nt, case.n_shots, case.rec.shape[1], device="cuda", dtype=dtype)
    bg_r = torch.zeros_like(r)
    fn = getattr(tide._native.load(),
                 f"maxwell_tm_{case.stencil}_{tide._native.dtype_name(dtype)}_born_forward_cuda")
    keep = [d(x) for x in (case.ca, case.cb, case.cq, dca, dcb, case.f, df)]
    prof = [d(x) for x in case.profiles]
    src, rec = (torch.from_numpy(np.ascontiguousarray(x)) for x in (case.src, case.rec))
    tide._native.check(fn(
        *[ptr(t) for t in (*keep, *bg, *sc, r, bg_r, *prof, src, rec)], case.rdy, case.rdx,
        case.dt, case.nt, case.n_shots, case.ny, case.nx, case.src.shape[1], case.rec.shape[1], 1,
        False, False, False, 0, *case.pml, 0, 0, tide._native.stream_handle(torch.device("cuda"))))
    torch.cuda.synchronize()
    return r.cpu().numpy(), bg_r.cpu().numpy(), [t.cpu().numpy() for t in bg]


@gpu
@pytest.mark.parametrize("stencil", [2, 4, 6, 8])
@pytest.mark.parametrize("ny,nx,nt", [(17, 130, 1), (49, 65, 7), (33, 49, 8), (40, 97, 17)])
def test_born_beside_the_tile_edges(stencil, ny, nx, nt):
    print(f"Born order {stencil} {ny}x{nx} nt {nt}", flush=True)
    for dtype in (torch.float64, torch.float32):
        case = _case(ny, nx, nt, stencil=stencil, dtype=dtype)
        rng = np.random.default_rng(1)
        dca = (1e-3 * rng.standard_normal((ny, nx))).astype(case.dtype)
        dcb = (1e-3 * np.abs(case.cb).mean() * rng.standard_normal((ny, nx))).astype(case.dtype)
        df = (1e-2 * np.abs(case.f).max() * rng.standard_normal(case.f.shape)).astype(case.dtype)
        f_o, r_f, _, _ = O.tm2d_forward(case)
        r_o, dr_o = O.tm2d_tangent(case.astype(np.float64), *(a.astype(np.float64)
                                                              for a in (dca, dcb, df)))
        dr, r, fields = _born(case, dca, dcb, df)
        assert np.array_equal(r, r_f)
        assert all(np.array_equal(a.reshape(b.shape), b) for a, b in zip(fields, f_o))
        if dtype == torch.float64:
            assert np.array_equal(r, r_o) and np.array_equal(dr, dr_o)
        else:  # rounding of at most 17 steps of about 20 fp32 operations each
            assert relative_l2(dr, dr_o) < 17 * 20 * 2.0**-24
        none, zero = _born(case, None, None, df), _born(case, 0 * dca, 0 * dcb, df)
        assert np.array_equal(none[0], zero[0]) and np.array_equal(none[1], r)


@gpu
@pytest.mark.parametrize("compression,interval,graph", [(False, 1, True), (False, 3, False),
                                                        (True, 2, True)])
def test_batched_plans_on_tiles(compression, interval, graph):
    _check_batch(compression, interval, graph)


def _check_batch(compression, interval, graph):
    """Problems of one and of several tiles and shots, whose loops take one
    launch, an even and an odd last launch: receivers, states and source
    gradients as the oracle's, replayed twice."""
    from tide.batch import TM2DBatch

    dev = torch.device("cuda:0")
    sizes = [(30, 44, 23, 2), (9, 8, 1, 1), (70, 121, 16, 3), (25, 90, 7, 11), (12, 33, 9, 1)]
    problems = []
    for ny, nx, nt, shots in sizes:
        g = torch.Generator().manual_seed(ny)
        dx = 0.01
        dt = 0.7 * dx / (2**0.5 * tide.C0)
        amp = tide.ricker(9e8, nt + 8, dt, peak_time=4 * dt)[:nt].reshape(1, 1, -1).repeat(shots, 2, 1)
        src = torch.stack([torch.tensor([[1 + s % (ny - 2), 2], [1 + s % (ny - 2), 2]])
                           for s in range(shots)])
        rec = torch.stack([torch.tensor([[2, x] for x in range(0, nx, 2)])] * shots)
        problems.append(dict(
            epsilon=(1 + 8 * torch.rand(ny, nx, generator=g)).to(dev),
            sigma=(0.01 * torch.rand(ny, nx, generator=g)).to(dev),
            mu=torch.ones(ny, nx, device=dev), grid_spacing=dx, dt=dt,
            source_amplitude=amp.to(dev), source_location=src.to(dev),
            receiver_location=rec.to(dev), pml_width=[3, 4, 5, 2]))
    batch = TM2DBatch(problems, storage_compression=compression, use_graph=graph,
                      model_gradient_sampling_interval=interval)
    store = "bf16" if compression else "full"
    cases = [O.case_from_setup(prepare_tm2d(**kw)) for kw in problems]
    rng = np.random.default_rng(4)
    for replay in range(2):
        batch.reset_state()
        rs = [r.cpu().numpy() for r in batch.forward()]
        ws = [rng.standard_normal(r.shape).astype(np.float32) for r in rs]
        states = [[t.cpu().numpy() for t in st.fields] for st in batch.setups]
        out = [[t.cpu().numpy() for t in ts]
               for ts in batch.backward([torch.from_numpy(w).to(dev) for w in ws])]
        for size, case, r, w, state, (ga, gb, gf) in zip(sizes, cases, rs, ws, states, out):
            print(f"replay {replay} problem {size}", flush=True)
            f_o, r_o, es, cs = O.tm2d_forward(case, store=store, interval=interval)
            assert np.array_equal(r, r_o)
            assert all(np.array_equal(a.reshape(b.shape), b) for a, b in zip(state, f_o))
            ga_o, gb_o, gf_o, _ = O.tm2d_backward(case, w, es, cs, store=store, interval=interval)
            assert np.array_equal(gf.reshape(gf_o.shape), gf_o)
            for a, b in ((ga, ga_o), (gb, gb_o)):
                assert relative_l2(a.reshape(b.shape), b) < 1e-12 if b.any() else not a.any()
    batch.close()


@pytest.fixture
def no_room():
    """Every tile loop of the test's thread finds its scratch too large."""
    lib = tide._native.load()
    lib.tide_tm2d_set_tile_scratch_limit(0)
    yield lib
    lib.tide_tm2d_set_tile_scratch_limit(-1)


@gpu
@pytest.mark.parametrize("stencil", [2, 4, 6, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_calls_without_room_for_tiles_fall_back(no_room, stencil, dtype):
    print(f"order {stencil} {dtype}", flush=True)
    _check(_case(49, 65, 13, stencil=stencil, dtype=dtype, shots=5))
    case = _case(33, 49, 9, stencil=stencil, dtype=dtype)
    rng = np.random.default_rng(1)
    dca = (1e-3 * rng.standard_normal((33, 49))).astype(case.dtype)
    dcb = (1e-3 * np.abs(case.cb).mean() * rng.standard_normal((33, 49))).astype(case.dtype)
    df = np.zeros_like(case.f)
    small = _born(case, dca, dcb, df)
    no_room.tide_tm2d_set_tile_scratch_limit(-1)
    tiles = _born(case, dca, dcb, df)
    assert np.array_equal(small[1], tiles[1])
    assert all(np.array_equal(a, b) for a, b in zip(small[2], tiles[2]))
    # the two sum the scattering term of a step in another order: rounding of 9
    # steps of about 20 operations
    assert relative_l2(small[0], tiles[0]) < 9 * 20 * np.finfo(case.dtype).eps


@gpu
@pytest.mark.parametrize("stencil", [2, 4])
def test_a_caller_that_can_make_room_is_told(no_room, stencil):
    """Without the fallback a call returns status 4, and the next is none the worse."""
    case = _case(40, 50, 9, stencil=stencil)
    no_room.tide_tm2d_set_tile_fallback(0)
    try:
        with pytest.raises(tide._native.TideNativeError, match="status 4"):
            gpu_forward(case)
        with pytest.raises(tide._native.TideNativeError, match="status 4"):
            gpu_forward(case, store="full")
        stores = np.zeros((case.nt, case.n_shots, case.ny, case.nx), case.dtype)
        w = np.ones((case.nt, case.n_shots, case.rec.shape[1]), case.dtype)
        with pytest.raises(tide._native.TideNativeError, match="status 4"):
            gpu_backward(case, w, stores, stores)
        with pytest.raises(tide._native.TideNativeError, match="status 4"):
            _born(case, None, None, np.zeros_like(case.f))
    finally:
        no_room.tide_tm2d_set_tile_fallback(1)
    no_room.tide_tm2d_set_tile_scratch_limit(-1)
    _check(case)  # an earlier call's failure is not a later one's


@gpu
@pytest.mark.parametrize("graph", [False, True])
def test_batched_plans_without_room_for_tiles_fall_back(no_room, graph):
    _check_batch(False, 1, graph)


@gpu
@pytest.mark.parametrize("blocks", [(0, 2), (0, 1), (2, 0), (1, 0), (0, 3)])
@pytest.mark.parametrize("compression,interval,graph", [(False, 1, True), (True, 2, False)])
def test_batched_plans_with_one_pass_on_tiles(blocks, compression, interval, graph):
    """Tiles in one pass, step launches in the other."""
    before = tide._native.get_tm2d_time_block()
    tide._native.set_tm2d_time_block(*blocks)
    try:
        _check_batch(compression, interval, graph)
    finally:
        tide._native.set_tm2d_time_block(*before)
