"""Stage kernels compiled for the terms a problem has (no source and a flat bed; Manning friction
alone) against the kernel that tests every term at run time.  A field that mixes 0.0 and -0.0
is stored point by point but changes no value, so it sends the same problem to the general
kernel: FP32 integrals must agree to the last bit (their rounding is fixed), FP64 to rounding
(1e-13 relative after two steps of values of order one)."""
import numpy as np
import pytest
import torch

from helpers import rel_l2
from oceano_amd import problems
from oceano_amd.integrator import AdditiveRungeKuttaIntegrator, DeviceIntegrator

pytestmark = pytest.mark.gpu


def _problem(kind, degree, split, signed_zeros):
    P = problems.vortex(degree=degree, refine=0, nx=18, ny=9, refine_fraction=split, seed=3)
    column = 0 if kind == "plain" else 2  # bed, wind

    def data(xy):
        out = np.zeros((xy.shape[0], 5))
        if kind == "manning":
            out[:, 0] = 0.05 * np.sin(np.pi * xy[:, 0])
            out[:, 1] = 0.03
        if signed_zeros:
            out[::2, column] = -0.0
        return out

    P.problem_data = data
    return P


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("split", [None, 0.3])
@pytest.mark.parametrize("degree", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["plain", "manning"])
def test_terms(cuda, kind, degree, split, precision):
    print("[terms] %s p=%d split=%s %s" % (kind, degree, split, precision), flush=True)
    out = []
    for signed_zeros in (False, True):
        P = _problem(kind, degree, split, signed_zeros)
        op, _, h, q = problems.setup_operator(P, precision=precision)
        rk = DeviceIntegrator(op)
        for _ in range(2):
            rk.step(2e-4, h, q)
        torch.cuda.synchronize()
        out.append((op.unpack(h, 1).cpu().numpy(), op.unpack(q, 2).cpu().numpy()))
    for a, b in zip(*out):
        if precision == "mixed":
            assert np.array_equal(a, b)
        else:
            assert rel_l2(a, b) <= 1e-13


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("split", [None, 0.3])
@pytest.mark.parametrize("degree", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["plain", "manning", "ark"])
def test_terms_of_one_evaluation(cuda, kind, degree, split, precision):
    """the same for dst = M^-1 L(src), L(src) and one additive step"""
    print("[terms] evaluation %s p=%d split=%s %s" % (kind, degree, split, precision), flush=True)
    out = []
    for signed_zeros in (False, True):
        P = _problem("plain" if kind == "plain" else "manning", degree, split, signed_zeros)
        op, _, h, q = problems.setup_operator(P, precision=precision)
        got = []
        if kind == "ark":
            rk = AdditiveRungeKuttaIntegrator()
            rk.reinit(op)
            rk.perform_time_step(op, 0.0, 2e-4, h, q)
            got = [h, q]
        else:
            for evaluate in (lambda d: op.apply(0.0, [h, q], d), lambda d: op.rhs([h, q], d)):
                dst = [torch.empty_like(h), torch.empty_like(q)]
                evaluate(dst)
                got += dst
        torch.cuda.synchronize()
        out.append([op.unpack(v, 1 + i % 2).cpu().numpy() for i, v in enumerate(got)])
    for a, b in zip(*out):
        if precision == "mixed":
            assert np.array_equal(a, b)
        else:  # M^-1 L of a smooth state is of order one; its terms cancel over 1/h ~ 50
            assert rel_l2(a, b) <= 1e-11
