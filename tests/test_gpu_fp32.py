"""FP32-bulk entry points (vls_sdf3_*_f32) against the FP64 path and the oracle.

Exact where the float path computes in FP64 on float inputs: setDistance
(subcell distances from F converted to double), the area/volume reductions and
the normal velocity equal the FP64 entry points on the same float values
converted to double.  Where the bulk arithmetic is FP32 (advection, extension,
reinitialization, surface redistance), the float result is compared with the
FP64 oracle started from the same float values, with the tolerance stated in
each test.
"""
import importlib

import numpy as np
import pytest
import torch

from golden import cases
from oracle import pyoracle as po

vls = importlib.import_module("2018_7_vesicle_amd")

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24  # FP32 unit roundoff


def _grid(n):
    g = cases.linspace_grid(n)
    return g, vls.GD3(g.xv, g.yv, g.zv)


def _f32(a):
    """a rounded to float32, as float64"""
    return np.ascontiguousarray(a, dtype=np.float32).astype(np.float64)


def _cuda(a, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


def _wobbly_sphere(g):
    r = np.sqrt(g.X ** 2 + g.Y ** 2 + g.Z ** 2)
    return (r - 0.6) * (1 + 0.2 * np.sin(3 * g.X) * np.cos(2 * g.Y))


def test_set_distance_f32_equals_fp64_on_same_values():
    g, G = _grid(40)
    F32 = _cuda(_wobbly_sphere(g), torch.float32)
    m32 = vls.SDF3(G, F32)
    m32.setDistance()
    d32 = [t.clone() for t in m32.distances()]
    m64 = vls.SDF3(G, F32.double())
    m64.setDistance()
    for a, b in zip(d32, m64.distances()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", [0, 1])
def test_area_volume_f32_equals_fp64_on_same_values(kind):
    g, G = _grid(36)
    F32 = _cuda(_wobbly_sphere(g), torch.float32)
    o32 = torch.zeros(2, dtype=torch.float64, device="cuda")
    o64 = torch.zeros(2, dtype=torch.float64, device="cuda")
    vls.SDF3(G, F32).areaVolumeDevice(o32, kind)
    vls.SDF3(G, F32.double()).areaVolumeDevice(o64, kind)
    assert torch.equal(o32, o64)


def test_normal_velocity_f32_is_rounded_fp64():
    g, G = _grid(32)
    F32 = _cuda(_wobbly_sphere(g), torch.float32)
    u32 = [_cuda(c, torch.float32) for c in cases.smooth_velocity(g)]
    out32 = torch.zeros_like(F32)
    vls.SDF3(G, F32).normalVelocity(*u32, out32)
    out64 = torch.zeros_like(F32, dtype=torch.float64)
    vls.SDF3(G, F32.double()).normalVelocity(*[c.double() for c in u32], out64)
    assert torch.equal(out32, out64.float())


def test_max_speed_f32():
    g, G = _grid(24)
    u32 = [_cuda(c, torch.float32) for c in cases.smooth_velocity(g)]
    m = vls.SDF3(G, _cuda(_wobbly_sphere(g), torch.float32))
    assert m.maxSpeed(*u32) == max(float(c.abs().max()) for c in u32)


def test_advection_f32_vs_oracle():
    """10 RK3 steps: within 300 FP32 roundings of max|F| of the FP64 oracle."""
    g, G = _grid(40)
    u = [_f32(c) for c in cases.smooth_velocity(g)]
    F0 = _f32(_wobbly_sphere(g))
    dt = 0.4 * g.dx / max(np.abs(c).max() for c in u)
    ref = po.advect_rk3(F0, 10, dt, u, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    out = m.WENO5RK3Advection(m.F, *[_cuda(c, torch.float32) for c in u], dt, 10).double().cpu().numpy()
    err = np.abs(out - ref).max() / np.abs(ref).max()
    assert err < 300 * U32, err


def test_reinit_f32_vs_oracle():
    """50 WENO5-RK3 reinitialization iterations in the band |phi| < 3 dx:
    within 1e-4 dx of the FP64 oracle, and the same sign at all but 1e-4 of
    the points."""
    g, G = _grid(40)
    F0 = _f32(_wobbly_sphere(g))
    d6, md = po.set_distance(F0, *g.spacing)
    ref = po.weno5_rk3_reinit(F0, 50, d6, md, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    m.setDistance()
    out = m.WENO5RK3Reinitialization(m.F, 50).double().cpu().numpy()
    band = np.abs(ref) < 3 * g.dx
    err = np.abs(out - ref)[band].max() / g.dx
    assert err < 1e-4, err
    assert np.mean((out < 0) != (ref < 0)) < 1e-4


def test_reinit_f32_fp64_tail_of_the_whole_call_is_the_fp64_result():
    """An FP64 tail as long as the call (vls_sdf3_set_reinit_fp64_tail): the
    FP32 call returns the FP64 oracle's result rounded to float, bit for bit."""
    g, G = _grid(40)
    F0 = _f32(_wobbly_sphere(g))
    d6, md = po.set_distance(F0, *g.spacing)
    ref = po.weno5_rk3_reinit(F0, 20, d6, md, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    m.setReinitFP64Tail(25)
    m.setDistance()
    out = m.WENO5RK3Reinitialization(m.F, 20).cpu().numpy()
    assert np.array_equal(out, ref.astype(np.float32))


def test_reinit_f32_fp64_tail_continues_the_fp32_iterations():
    """A 30-iteration FP32 call with a 10-iteration FP64 tail is the 20 FP32
    iterations followed by 10 FP64 iterations with the call's mask and
    distances (those of the input): against the oracle continuing the FP32
    result, bit for bit after rounding to float."""
    g, G = _grid(40)
    F0 = _f32(_wobbly_sphere(g))
    d6, md = po.set_distance(F0, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    m.setDistance()
    a = m.WENO5RK3Reinitialization(m.F.clone(), 20).double().cpu().numpy()
    # the oracle takes its mask from its input: the continuation is exact when
    # the FP32 iterations kept every sign
    assert np.array_equal(a < 0, F0 < 0)
    ref = po.weno5_rk3_reinit(a, 10, d6, md, *g.spacing)
    m.setReinitFP64Tail(10)
    out = m.WENO5RK3Reinitialization(m.F, 30).cpu().numpy()
    assert np.array_equal(out, ref.astype(np.float32))


def test_extend_f32_vs_oracle():
    """40 WENO5-RK3 extension iterations off a sphere: within 1e-5 of max|C|."""
    g, G = _grid(40)
    F0 = _f32(np.sqrt(g.X ** 2 + g.Y ** 2 + g.Z ** 2) - 0.55)
    C = _f32(np.sin(2 * g.X) + g.Y * g.Z)
    d6, md = po.set_distance(F0, *g.spacing)
    ref = po.weno5_rk3_extend(C, 40, F0, d6, md, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    m.setDistance()
    out = m.WENO5RK3Extend(_cuda(C, torch.float32), 40).double().cpu().numpy()
    err = np.abs(out - ref).max() / np.abs(C).max()
    assert err < 1e-5, err


def test_surface_redistance_f32_vs_oracle():
    """(4, 3) closest-point surface redistance: within 1e-4 of the FP64 oracle
    in the band |F| < 3 dx."""
    g, G = _grid(32)
    F0 = _f32(np.sqrt(g.X ** 2 + g.Y ** 2 + g.Z ** 2) - 0.6)
    A = _f32(np.exp(g.Z) - 1)
    ref = po.surface_redistance(A, F0, 4, 3, *g.spacing)
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    out = m.WENO5RK3ClosetPointSurfaceRedistance(_cuda(A, torch.float32), 4, 3).double().cpu().numpy()
    band = np.abs(F0) < 3 * g.dx
    err = np.abs(out - ref)[band].max()
    assert err < 1e-4, err


@pytest.mark.parametrize("amplitude", [1.0, 1e5, 1e6, 3e6])
def test_fp32_operators_on_large_rough_fields(amplitude):
    """One advection step, one reinitialization iteration and one extension
    iteration of fields of independent random values of `amplitude`, whose second
    differences are as large, on spacings of 0.1 and without an interface (beside
    one, subcells of almost no width make random values ill-conditioned): the
    WENO weights, which fall as the fourth power of the differences, keep their
    accuracy.  A step adds at most a third of the correction Q to a value
    (Courant number 0.3 over 12 and three axes and stages), whose error is
    below 1e-5 of the amplitude, and a few roundings of the value: 64 FP32
    roundings of the amplitude."""
    rng = np.random.default_rng(11)
    g = cases.Grid(*[(np.arange(k) - (k - 1) / 2) * h for k, h in ((21, 0.1), (35, 0.09), (20, 0.11))])
    G = vls.GD3(g.xv, g.yv, g.zv)
    rough = _f32(amplitude * rng.uniform(-1, 1, g.shape))
    lifted = _f32(amplitude * (3 + rng.uniform(-1, 1, g.shape)))
    u = [_f32(rng.uniform(-1, 1, g.shape)) for _ in range(3)]
    F0 = _f32(0.7 * g.X + 0.5 * g.Y - 0.6 * g.Z + 9.0)
    errs = {}

    def check(name, out, ref):
        errs[name] = np.abs(out.double().cpu().numpy() - ref).max() / amplitude

    m = vls.SDF3(G, _cuda(rough, torch.float32))
    check("advect", m.WENO5RK3Advection(m.F, *[_cuda(c, torch.float32) for c in u], 0.02, 1),
          po.advect_rk3(rough, 1, 0.02, u, *g.spacing))
    m = vls.SDF3(G, _cuda(lifted, torch.float32))
    m.setDistance()
    d6, md = po.set_distance(lifted, *g.spacing)
    check("reinit", m.WENO5RK3Reinitialization(m.F, 1), po.weno5_rk3_reinit(lifted, 1, d6, md, *g.spacing))
    m = vls.SDF3(G, _cuda(F0, torch.float32))
    m.setDistance()
    d6, md = po.set_distance(F0, *g.spacing)
    check("extend", m.WENO5RK3Extend(_cuda(rough, torch.float32), 1),
          po.weno5_rk3_extend(rough, 1, F0, d6, md, *g.spacing))
    assert all(e < 64 * U32 for e in errs.values()), errs


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_reinit_rounds_alike_on_every_axis(dtype, sign):
    """A line of 1000 random values, constant across, reinitialized with the
    line laid along x, y and z: the same bits (the z axis carries half of its
    weights from page to page, the other two do not)."""
    n, w = 1000, 4
    f = sign * np.random.default_rng(3).uniform(0.001, 2.0, n)
    outs = []
    for dim in (1, 2, 0):  # x, y, z of a (pges, cols, rows) field
        shape = [w, w, w]
        shape[dim] = n
        pges, cols, rows = shape
        line = [1, 1, 1]
        line[dim] = n
        m = vls.SDF3(vls.GD3(*[np.arange(k) / 16 for k in (cols, rows, pges)]),
                     _cuda(np.broadcast_to(f.reshape(line), shape), dtype))
        m.setDistance()
        out = m.WENO5RK3Reinitialization(m.F, 10).movedim(dim, 0).reshape(n, w * w)
        assert torch.equal(out, out[:, :1].expand(n, w * w))
        outs.append(out[:, 0])
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_fp32_rejects_fp64_only_methods():
    g, G = _grid(16)
    m = vls.SDF3(G, _cuda(_wobbly_sphere(g), torch.float32))
    with pytest.raises(vls.VLSError):
        m.ENORK2Reinitialization(m.F, 1)
    with pytest.raises(vls.VLSError):
        m.WENO5RK3Reinitialization(m.F.double(), 1)
