"""The FP64 operators on boxes of very small and very large spacings, against
the oracle, bit for bit: the quotients of the WENO weights and of the
nonuniform stencils are computed without operand scaling (quot in
vls_device.hpp), so their numerators and denominators follow the spacing's
scale over its eighth power."""
import importlib

import numpy as np
import pytest
import torch

import cases
from oracle import pyoracle as po

vls = importlib.import_module("2018_7_vesicle_amd")
pytestmark = pytest.mark.gpu


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", torch.float64)


@pytest.mark.parametrize("scale", [1e-12, 1e-3, 1e10])
def test_operators_at_a_scale(scale):
    g1 = cases.Grid(np.linspace(-1.0, 1.0, 19), np.linspace(-0.95, 0.95, 35), np.linspace(-1.05, 1.05, 17))
    F = np.ascontiguousarray(cases.star_phi0(g1) * scale)
    C = np.ascontiguousarray(cases.smooth_scalar(g1))
    g = cases.Grid(g1.xv * scale, g1.yv * scale, g1.zv * scale)
    G = vls.GD3(g.xv, g.yv, g.zv)
    m = vls.SDF3(G, T(F))
    m.setDistance()
    d6, md = po.set_distance(F, *g.spacing)
    got = {
        "reinit": (m.WENO5RK3Reinitialization(T(F), 3), po.weno5_rk3_reinit(F, 3, d6, md, *g.spacing)),
        "extend": (m.WENO5RK3Extend(T(C), 3), po.weno5_rk3_extend(C, 3, F, d6, md, *g.spacing)),
        "advect": (m.WENO5RK3Advection(T(F), *[T(u * scale) for u in cases.smooth_velocity(g1)], 0.01, 2),
                   po.advect_rk3(F, 2, 0.01, [u * scale for u in cases.smooth_velocity(g1)], *g.spacing)),
        "cubic reinit": (m.WENORK3Reinitialization(T(F), 3), po.wenork3_reinit(F, 3, *g.spacing)),
        "cubic extend": (m.WENORK3Extend(T(C), 3), po.variant_extend(C, 3, F, *g.spacing, "wenork3")),
        "eno2 reinit": (m.ENORK2Reinitialization(T(F), 3), po.eno2_reinit(F, 3, *g.spacing)),
        "eno2 extend": (m.ENORK2Extend(T(C), 3), po.variant_extend(C, 3, F, *g.spacing, "enork2")),
    }
    for name, (a, ref) in got.items():
        assert np.array_equal(a.cpu().numpy(), ref), f"{name} at {scale}: {np.abs(a.cpu().numpy() - ref).max():.2e}"
