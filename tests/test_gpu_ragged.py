"""Sizes around the tiles of the kernels that move or map whole tiles: pack / unpack (64 cells
through LDS) and the closure network (16 samples a wave, 64 a workgroup), at remainders and at
the smallest calls."""
import numpy as np
import pytest
import torch

import mlp_oracle as mo
from helpers import rel_l2, to_host
from oceano_amd import closure, problems
from oceano_amd.mlp import ClosureNetwork

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 1), (9, 7), (8, 8), (13, 5), (64, 2), (43, 3)])
@pytest.mark.parametrize("degree", [1, 2, 3, 4])
def test_pack_round_trip(cuda, degree, nx, ny):
    """unpack(pack(x)) is x bit for bit; every value is stored once"""
    print("[ragged] pack p=%d cells=%d" % (degree, nx * ny), flush=True)
    P = problems.vortex(degree=degree, refine=0, nx=nx, ny=ny)
    op, _, _, _ = problems.setup_operator(P)
    rng = np.random.default_rng(degree)
    for nc in (1, 2):
        x = rng.standard_normal(nx * ny * nc * (degree + 1) ** 2)
        v = op.pack(x, nc)
        assert np.array_equal(op.unpack(v, nc).cpu().numpy(), x)
        stored = np.isin(v.cpu().numpy(), x).sum()
        assert stored == x.size


def _net(seed):
    net = ClosureNetwork(30, 18, seed=seed)
    rng = np.random.default_rng(seed)
    net.set_normalization(rng.standard_normal(30) * 0.2, 0.5 + rng.random(30),
                          rng.standard_normal(18) * 0.1, 0.5 + rng.random(18))
    ref = mo.Network(net.get_params().astype(np.float64), 30, 18, norm=net.normalization)
    return net, ref, rng


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4097])
def test_network_rows(cuda, n):
    """The sums of a product are taken in another order than the oracle's, which can round an
    activation to the neighbouring BF16 value (2^-8 relative), once in each of four layers:
    2^-6 for a single sample's gradient, and the forward values within that."""
    print("[ragged] network rows=%d" % n, flush=True)
    net, ref, rng = _net(21)
    x = rng.standard_normal((n, 30)).astype(np.float32)
    t = (rng.standard_normal((n, 18)) * 0.3).astype(np.float32)
    X, T = torch.tensor(x, device=cuda), torch.tensor(t, device=cuda)
    y = net.forward(X).cpu().numpy()
    assert y.shape == (n, 18)
    assert rel_l2(y, ref.predict(x.astype(np.float64))) < 2.0 ** -6
    loss, g = net.gradients(X, T)
    lref, gref = ref.loss_and_gradient(x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - lref) < 2.0 ** -6 * lref
    assert rel_l2(g, gref) < 2.0 ** -6


@pytest.mark.parametrize("nx,ny", [(3, 1), (17, 1), (32, 2), (33, 2), (81, 1)])
def test_closure_cells(cuda, nx, ny):
    """the correction of every cell of a mesh whose last tile is partly filled"""
    print("[ragged] closure cells=%d" % (nx * ny), flush=True)
    S = closure.SubgridChannel(1003, nx=nx, ny=ny, factor=2)
    op, _, h, q = problems.setup_operator(S.plain)
    op.set_subgrid_stats(S.cell_stats(S.plain.mesh))
    net, ref, _ = _net(13)
    op.set_closure(net)
    tau = op.closure_source(h, q)
    tm = ref.predict(op.closure_features(h, q).cpu().numpy().astype(np.float64))
    _, V = closure.nodal_to_modal(2)
    want = np.stack([tm[:, :9] @ V.T, tm[:, 9:] @ V.T], 1).ravel()
    assert rel_l2(to_host(op, tau, 2), want) < 2.0 ** -6
