"""Viscous stage kernels compiled for the terms a problem has against the one that tests every term
at run time: a field that mixes 0.0 and -0.0 is stored but changes no value, and sends the same
problem there.  FP32 integrals must agree to the last bit (their rounding is fixed), FP64 to
rounding (1e-13 relative after two steps of values of order one)."""
import numpy as np
import pytest
import torch

from helpers import rel_l2
from oceano_amd import problems
from oceano_amd.integrator import DeviceIntegrator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("split", [None, 0.3])
@pytest.mark.parametrize("degree", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["plain", "manning"])
def test_terms_of_the_viscous_stage(cuda, kind, degree, split, precision):
    print("[terms] viscous %s p=%d split=%s %s" % (kind, degree, split, precision), flush=True)
    out = []
    for signed_zeros in (False, True):
        P = problems.vortex(degree=degree, refine=0, nx=18, ny=9, refine_fraction=split, seed=3)
        P.viscosity = 1e-3

        def data(xy):
            d = np.zeros((xy.shape[0], 5))
            if kind == "manning":
                d[:, 0] = 0.05 * np.sin(np.pi * xy[:, 0])
                d[:, 1] = 0.03
            if signed_zeros:
                d[::2, 2 if kind == "manning" else 0] = -0.0
            return d

        P.problem_data = data
        op, _, h, q = problems.setup_operator(P, precision=precision)
        rk, vel = DeviceIntegrator(op), op.velocity(h, q)
        for _ in range(2):
            rk.step(2e-4, h, q, vel)
        torch.cuda.synchronize()
        out.append((op.unpack(h, 1).cpu().numpy(), op.unpack(q, 2).cpu().numpy()))
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        if precision == "mixed":
            assert np.array_equal(a, b)
        else:
            assert rel_l2(a, b) <= 1e-13
