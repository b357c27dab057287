"""FP64 Manning powers (h^-1/3 of the source, h^-4/3 of its Jacobian) over the range of depths,
against the CPU oracle: one additive stage of a uniform flow over a flat periodic bed.  Its
stiff k vector is the friction source tested against the basis and nothing else
(OceanDG.h:794-826), its next stage input is divided by 1 + fm J (OceanDG.h:1574-1645).

Tolerances: the k vector is a sum of terms of one sign, each a product of a dozen factors good
to two ulp; the oracle's exp(a log h) adds a |ln h| ulp (|ln h| <= 21 here): 1e-14.  The update
is good to 1e-12 as every stage output."""
import numpy as np
import pytest
import torch

from helpers import rel_l2
from oceano_amd import problems
from oceano_amd.integrator import ark_tableau
from oceano_amd.mesh import Mesh
import pyoracle

pytestmark = pytest.mark.gpu


def _uniform(depth, degree):
    mesh = Mesh.rectangle(0.0, 2.0, 0.0, 1.0, 10, 5, periodic=(True, True))

    def data(xy):
        out = np.zeros((xy.shape[0], 5))
        out[:, 0], out[:, 1] = depth, 3.0
        return out

    def initial(xy):
        return np.tile([0.0, 0.7, -0.4], (xy.shape[0], 1))

    return problems.Problem(mesh, degree, {}, data, initial, name="uniform")


@pytest.mark.parametrize("degree", [1, 3])
@pytest.mark.parametrize("depth", [1e-9, 1e-4, 0.09, 0.11, 0.5, 0.999, 1.0, 2.0, 37.0, 1e3, 1e5])
def test_friction_powers(cuda, depth, degree):
    print("[manning] depth=%g p=%d" % (depth, degree), flush=True)
    P = _uniform(depth, degree)
    op, _, _, _ = problems.setup_operator(P)
    o = pyoracle.Oracle.from_mesh(P.mesh, degree)
    data = o.initialize_data_at_quadrature(P.problem_data)
    h, q = o.project_hydro(P.initial, data["cell_2"][:, 0])
    gh, gq = op.pack(h, 1), op.pack(q, 2)
    a, _, _, at, d = ark_tableau()
    dt = 1e-3
    kh, kq = [o.zeros(1) for _ in range(4)], [o.zeros(2) for _ in range(6)]
    rh, rq = o.zeros(1), o.zeros(2)
    o.perform_stage_hydro_ark(0, 3, np.array(a[0]) * dt, np.array(at[0]) * dt, d[0] * dt, h, q,
                              None, kh, kq, h, q, rh, rq)
    gkh = [op.initialize_vector(0) for _ in range(4)]
    gkq = [op.initialize_vector(1) for _ in range(6)]
    grh, grq = op.initialize_vector(0), op.initialize_vector(1)
    op.perform_stage_hydro_ark(0, 0.0, np.array(a[0]) * dt, np.array(at[0]) * dt, d[0] * dt,
                               [gh, gq], gkh, gkq, gh, gq, grh, grq)
    torch.cuda.synchronize()
    assert rel_l2(op.unpack(gkq[2], 2).cpu().numpy(), kq[2]) <= 1e-14
    assert rel_l2(op.unpack(grq, 2).cpu().numpy(), rq) <= 1e-12
