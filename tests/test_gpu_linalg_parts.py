"""The subspace projection where its rows are split over the wavefronts of a
workgroup: part sizes that end inside a step, parts without rows, one to
several tiles per workgroup; and products staged one after another through
the same host memory."""
import numpy as np
import pytest

from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    cfg, ints, _ = inputs.workload("fci6")
    H = api.Hamiltonian(cfg, ints)
    yield H
    H.close()


@pytest.mark.parametrize("m,b", [(1, 1), (16, 16), (17, 3), (33, 17), (64, 16), (65, 33)])
@pytest.mark.parametrize("n", [1, 63, 64, 513, 16383, 131073, 300001])
def test_project_parts(ctx, n, m, b):
    import torch
    g = torch.Generator().manual_seed(n + 7 * m + b)
    A = torch.randn(n, m + 3, generator=g, dtype=torch.float64)
    B = torch.randn(n, b + 1, generator=g, dtype=torch.float64)
    ref = A[:, :m].numpy().T @ B[:, 1:].numpy()
    out = ctx.project(A.cuda()[:, :m], B.cuda()[:, 1:])
    # sums of n products of unit variance
    assert np.abs(out - ref).max() <= 1e-14 * max(n, 64), np.abs(out - ref).max()


def test_staged_products_in_turn(ctx):
    import torch
    rng = np.random.default_rng(4)
    n = 4099
    A = rng.standard_normal((n, 96))
    Ad = torch.from_numpy(A).cuda()
    O = torch.zeros(n, 96, dtype=torch.float64, device="cuda")
    want = np.zeros((n, 96))
    # more small matrices (0.07 MB each) than the staging memory holds
    for i in range(12):
        Y = rng.standard_normal((96, 96))
        ctx.combine(Ad, Y, O, 0.5)
        want = 0.5 * want + A @ Y
    assert np.abs(O.cpu().numpy() - want).max() <= 1e-11 * np.abs(want).max()
