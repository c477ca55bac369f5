"""FP64 reinitialization of a field that changes sign at nearly every point: a
block of the stage lists its bulk points beside a sign change (up to all 256
points of its 16 pages) and evaluates them after its march.  Against the oracle,
bit for bit, at depths below, at and above the pages such a block takes."""
import importlib

import numpy as np
import pytest
import torch

import cases
from oracle import pyoracle as po

vls = importlib.import_module("2018_7_vesicle_amd")
bm = importlib.import_module("2018_7_vesicle_amd.batch")
pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", torch.float64)


def _problem(rows, cols, pges):
    g = cases.Grid(np.linspace(-1.0, 1.0, cols), np.linspace(-0.95, 0.95, rows), np.linspace(-1.05, 1.05, pges))
    F = np.ascontiguousarray(cases.star_phi0(g))
    p, c, r = np.meshgrid(np.arange(pges), np.arange(cols), np.arange(rows), indexing="ij")
    A = np.ascontiguousarray(np.sin(1.7 * r + 0.3) * np.cos(1.3 * c + 0.9 * p) * g.spacing[0])
    d6, md = po.set_distance(F, *g.spacing)
    return g, F, A, po.weno5_rk3_reinit(A, 1, d6, md, *g.spacing)


@pytest.mark.parametrize("rows", [32, 64])
@pytest.mark.parametrize("depth", [3, 16, 17, 40])
def test_single_grid(rows, depth):
    g, F, A, ref = _problem(rows - 3, 19, 41)
    m = vls.SDF3(vls.GD3(g.xv, g.yv, g.zv), T(F))
    m.setTileRows(rows)
    m.setZmarchDepth(depth)
    m.setDistance()
    got = m.WENO5RK3Reinitialization(T(A), 1).cpu().numpy()
    assert np.array_equal(got, ref), np.abs(got - ref).max()


@pytest.mark.parametrize("depth", [1, 16, 17, 40])
def test_batch(depth):
    probs = [_problem(29, 19, 41), _problem(9, 33, 7), _problem(35, 10, 17)]
    b = bm.Batch([(q[0].rows, q[0].cols, q[0].pges) for q in probs], [q[0].spacing for q in probs], torch.float64)
    b.zmarch_depth = depth
    F, A = b.pack([T(q[1]) for q in probs]), b.pack([T(q[2]) for q in probs])
    b.set_distance(F)
    b.reinitialize(A, 1)
    for i, q in enumerate(probs):
        got = b.grid_view(A, i).cpu().numpy()
        assert np.array_equal(got, q[3]), (i, np.abs(got - q[3]).max())


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 5, 3), (16, 16, 5), (17, 31, 4)])
def test_point_kernels_with_every_axis_beside_a_crossing(shape):
    """the drop-ins whose blocks list their long evaluations: all three axes (six
    sides) of every point of a block, on boxes of less than a block, of whole
    blocks and of ragged ones; some points frozen, some sides at the spacing"""
    rows, cols, pges = shape
    sp = (0.11, 0.07, 0.13)
    rng = np.random.default_rng(rows * cols)
    p, c, r = np.meshgrid(np.arange(pges), np.arange(cols), np.arange(rows), indexing="ij")
    F = np.ascontiguousarray(np.where((r + c + p) % 2, 1.0, -1.0) * rng.uniform(0.2, 1.0, r.shape) * sp[0])
    C = rng.normal(size=F.shape)
    d6 = [h * rng.choice([1.0, 0.9, 0.4, 1e-9], p=[0.2, 0.4, 0.39, 0.01], size=F.shape)
          for h in np.repeat(sp, 2)]
    vel = [rng.normal(size=F.shape) for _ in range(3)]
    dt = 0.3 * np.min(np.stack(d6), axis=0)
    mask = (F < 0).astype(np.uint8)
    geo, n, d = (rows, cols, pges, *sp), F.size, [T(a) for a in d6]
    empty = lambda k: [torch.full(F.shape, np.nan, dtype=torch.float64, device="cuda") for _ in range(k)]  # noqa: E731

    loc, loc_ref = [T(a) for a in po.prefilled_distances(F.shape, *sp)], po.prefilled_distances(F.shape, *sp)
    po.boundary_location(loc_ref, F, *sp)
    vls.feval_boundary_location(*loc, T(F), n, *geo)
    step, cp, ext, nrm = empty(1), empty(6), empty(1), empty(3)
    vls.feval_re_step(step[0], T(F), T(mask).to(torch.uint8), T(dt), *d, *geo, n)
    vls.feval_upwind_normal(*nrm, T(F), *d, *geo, n)
    vls.feval_boundary_interpolant(*cp, *d, T(C), *geo, n)
    cp_ref = po.boundary_interpolant(d6, C, *sp)
    vls.feval_extend_step(ext[0], T(dt), T(C), *[T(a) for a in vel], *d, *[T(a) for a in cp_ref], *geo, n)
    for name, got, ref in (("distance", loc, loc_ref), ("re_step", step, [po.re_step(F, mask, dt, d6, *sp)]),
                           ("normal", nrm, po.upwind_normal(F, d6, *sp)), ("interpolant", cp, cp_ref),
                           ("extend_step", ext, [po.extend_step(dt, C, vel, d6, cp_ref, *sp)])):
        for k, (a, b) in enumerate(zip(got, ref)):
            assert np.array_equal(a.cpu().numpy(), b), (name, k)


def test_upwind_normal_at_any_distance():
    """upwind_normal takes distances down to zero (re_step and extend_step freeze
    a point below 1e-6 of the spacing): a cell of almost no width drops out of
    the weights where its squares overflow, and a zero distance gives NaN"""
    sp = (0.11, 0.07, 0.13)
    rng = np.random.default_rng(5)
    F = rng.normal(size=(5, 9, 33))
    d6 = [h * rng.choice([1.0, 0.4, 1e-16, 1e-120, 1e-160, 1e-200, 1e-300, 1e-310, 0.0], size=F.shape)
          for h in np.repeat(sp, 2)]
    nrm = [torch.full(F.shape, 7.0, dtype=torch.float64, device="cuda") for _ in range(3)]
    vls.feval_upwind_normal(*nrm, T(F), *[T(a) for a in d6], 33, 9, 5, *sp, F.size)
    for k, (a, b) in enumerate(zip(nrm, po.upwind_normal(F, d6, *sp))):
        assert np.isfinite(b).any()
        assert np.array_equal(a.cpu().numpy(), b, equal_nan=True), k


def test_extend_step_beside_huge_values():
    """extend_step at interface points some of whose stencils reach a value of
    1e200: the products of their divided differences overflow, and the stencil
    gets no weight where the oracle gives it none (NaN where the oracle has it)"""
    shape, sp = (5, 9, 33), (0.11, 0.07, 0.13)
    rng = np.random.default_rng(8)
    C = rng.normal(size=shape)
    C = np.where(rng.uniform(size=shape) < 0.03, 1e200 * C, C)
    d6 = [np.ascontiguousarray(h * rng.choice([1.0, 0.9, 0.4], size=shape)) for h in np.repeat(sp, 2)]
    vel = [rng.normal(size=shape) for _ in range(3)]
    cp6 = [rng.normal(size=shape) for _ in range(6)]
    dt = 0.3 * np.min(np.stack(d6), axis=0)
    ref = po.extend_step(dt, C, vel, d6, cp6, *sp)
    ext = torch.full(shape, 7.0, dtype=torch.float64, device="cuda")
    vls.feval_extend_step(ext, T(dt), T(C), *[T(a) for a in vel], *[T(a) for a in d6], *[T(a) for a in cp6],
                          33, 9, 5, *sp, C.size)
    assert np.array_equal(ext.cpu().numpy(), ref, equal_nan=True)


@pytest.mark.parametrize("shape", [(53, 8, 3), (54, 8, 3), (191, 8, 2), (192, 4, 2), (193, 4, 2), (500, 8, 3),
                                   (500, 7, 2), (1021, 43, 2)])
def test_point_kernels_on_either_walk(shape):
    """the boxes where the point kernels change between pages in memory order and
    64 x 4 tiles (from 192 rows on if they fit within 5%; advection_step within
    20%), with whole tiles and with ragged ones"""
    test_point_kernels_with_every_axis_beside_a_crossing(shape)
    rows, cols, pges = shape
    sp = (0.11, 0.07, 0.13)
    rng = np.random.default_rng(rows)
    F, *vel = [rng.normal(size=(pges, cols, rows)) for _ in range(4)]
    out = torch.full(F.shape, np.nan, dtype=torch.float64, device="cuda")
    vls.feval_advection_step(out, *[T(a) for a in vel], T(F), rows, cols, pges, *sp)
    assert np.array_equal(out.cpu().numpy(), po.advection_step(vel, F, *sp))
