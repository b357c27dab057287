"""FP64 degree 4 on meshes with hanging faces, with kernels of other degrees and precisions run before
every evaluation: no result may depend on what a register or LDS word held before.  Bar of the
parity tests, relative L2 <= 1e-12."""
import numpy as np
import pytest
import torch

from helpers import make_pair, rel_l2, to_dev, to_host
from oceano_amd import problems, tune
from oceano_amd.integrator import butcher_rows

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def others(cuda):
    """runs M^-1 L, L and a stage of degrees 1, 3 and 4 in both precisions, on other data"""
    ops = []
    for degree in (1, 3, 4):
        for precision in ("fp64", "mixed"):
            P = problems.vortex(degree=degree, refine=0, nx=40, ny=20, refine_fraction=0.4,
                                seed=degree)
            op, _, h, q = problems.setup_operator(P, precision=precision)
            vectors = [[op.initialize_vector(c) for c in (0, 1)] for _ in range(5)]
            ops.append((op, h, q, vectors))

    def run():
        for op, h, q, (d, k0, k1, w, r) in ops:
            op.apply(0.0, [h, q], d)
            op.rhs([h, q], d)
            w[0].copy_(h)
            w[1].copy_(q)
            op.perform_stage_hydro(0, 0.0, [1e-5], [h, q, None, None], [k0[0], k1[0]],
                                   [k0[1], k1[1]], w[0], w[1], r[0], r[1])
    return run


def _problem(kind, split):
    P = problems.vortex(degree=4, refine=0, nx=11, ny=7, refine_fraction=split,
                        seed=int(split * 10))
    base = P.problem_data

    def data(xy):
        out = base(xy)
        if kind != "plain":
            out[:, 0] = 0.05 * np.sin(np.pi * xy[:, 0])
            out[:, 1] = 0.03
        if kind == "general":
            out[:, 2] = 0.01
            out[:, 4] = 0.1
        return out

    P.problem_data = data
    return P


def _state(o, h, q):
    rng = np.random.default_rng(7)
    return h + 1e-3 * rng.standard_normal(h.shape), q + 1e-2 * rng.standard_normal(q.shape)


@pytest.mark.parametrize("kind", ["plain", "manning", "general"])
@pytest.mark.parametrize("split", [0.1, 0.4, 0.8])
def test_evaluations(cuda, others, split, kind):
    print("[between] evaluations split=%g %s" % (split, kind), flush=True)
    op, o, h, q = make_pair(_problem(kind, split))
    h, q = _state(o, h, q)
    L = o.rhs(h, q)
    M = [o.inverse_mass_tensor(L[0], 1), o.inverse_mass_tensor(L[1], 2)]
    src = [to_dev(op, h, 1), to_dev(op, q, 2)]
    for _ in range(2):
        for evaluate, want in ((lambda d: op.rhs(src, d), L),
                               (lambda d: op.apply(0.0, src, d), M)):
            others()
            dst = [op.initialize_vector(0), op.initialize_vector(1)]
            evaluate(dst)
            assert rel_l2(to_host(op, dst[0], 1), want[0]) <= TOL
            assert rel_l2(to_host(op, dst[1], 2), want[1]) <= TOL


@pytest.mark.parametrize("kind", ["plain", "manning", "general"])
@pytest.mark.parametrize("pair", [0, 1])
def test_stages(cuda, others, pair, kind):
    print("[between] stages paired_items=%d %s" % (pair, kind), flush=True)
    tune.apply_options({"paired_items": pair})
    try:
        op, o, h, q = make_pair(_problem(kind, 0.4))
    finally:
        tune.apply_options({"paired_items": -1})
    h, q = _state(o, h, q)
    rows, _ = butcher_rows("stage_4_order_4", 1e-4)
    S = len(rows)
    w_h, w_q, k_h, k_q = h.copy(), q.copy(), [o.zeros(1) for _ in range(S + 1)], \
        [o.zeros(2) for _ in range(S + 1)]
    o.time_step(rows, w_h, w_q, k_h, k_q, o.zeros(1), o.zeros(2))
    gw = [to_dev(op, h, 1), to_dev(op, q, 2)]
    gk = [[op.initialize_vector(c) for _ in range(S + 1)] for c in (0, 1)]
    gr = [[op.initialize_vector(0), op.initialize_vector(1)] for _ in range(2)]
    for s in range(S):
        others()
        src = gw if s == 0 else gr[s % 2]
        nxt = gr[(s + 1) % 2]
        op.perform_stage_hydro(s, 0.0, rows[s][:s + 1], src + [None, None], gk[0], gk[1],
                               gw[0], gw[1], nxt[0], nxt[1], write_scratch=True)
    torch.cuda.synchronize()
    assert rel_l2(to_host(op, gw[0], 1), w_h) <= TOL
    assert rel_l2(to_host(op, gw[1], 2), w_q) <= TOL
    for j in range(S + 1):
        assert rel_l2(to_host(op, gk[0][j], 1), k_h[j]) <= TOL
        assert rel_l2(to_host(op, gk[1][j], 2), k_q[j]) <= TOL
