"""FP64 MFMA subspace projection (A^T B over n rows) against numpy, for the
shapes the Davidson uses: tall-skinny, ragged tiles, column offsets."""
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


@pytest.mark.parametrize("n,m,b,ld", [(246, 4, 4, 20), (246, 20, 3, 20), (31650, 37, 17, 40), (100003, 80, 16, 96),
                                      (5, 1, 1, 1)])
def test_project_matches_numpy(ctx, n, m, b, ld):
    import torch
    g = torch.Generator().manual_seed(n + m)
    A = torch.randn(n, ld, generator=g, dtype=torch.float64)
    B = torch.randn(n, ld, generator=g, dtype=torch.float64)
    ref = A[:, :m].numpy().T @ B[:, ld - b:].numpy()
    Ad = A.cuda()
    Bd = B.cuda()
    out = ctx.project(Ad[:, :m], Bd[:, ld - b:])
    assert np.abs(out - ref).max() <= 1e-12 * max(1.0, np.abs(ref).max()), np.abs(out - ref).max()


@pytest.mark.parametrize("n,m,k,lda,ldo,alpha", [(246, 4, 4, 20, 4, 0.0), (246, 20, 3, 20, 7, 1.0),
                                                 (31650, 37, 17, 40, 17, 0.0), (100003, 120, 24, 120, 24, 0.0),
                                                 (100003, 120, 48, 120, 48, -0.5), (5, 1, 1, 1, 1, 2.0),
                                                 (4097, 130, 129, 130, 140, 1.0)])
def test_combine_matches_numpy(ctx, n, m, k, lda, ldo, alpha):
    """The MFMA basis update Out = alpha Out + A Y: ragged row tiles, t
    chunks and column tiles (k up to 129: two column slices)."""
    import torch
    g = torch.Generator().manual_seed(n + m + k)
    A = torch.randn(n, lda, generator=g, dtype=torch.float64)
    O = torch.randn(n, ldo, generator=g, dtype=torch.float64)
    Y = np.random.default_rng(m).standard_normal((m, k))
    ref = O.numpy().copy()
    ref[:, :k] = alpha * ref[:, :k] + A[:, :m].numpy() @ Y
    Od = O.cuda()
    ctx.combine(A.cuda()[:, :m], Y, Od[:, :k], alpha)
    out = Od.cpu().numpy()
    scale = max(1.0, np.abs(ref).max())
    assert np.abs(out - ref).max() <= 1e-12 * scale * max(1.0, m / 16)


def test_large_small_matrices(ctx):
    """Matrices beyond the pinned staging (more than 4 MiB) and at its edge."""
    import torch
    g = torch.Generator().manual_seed(5)
    n = 700
    for m in (724, 725, 900):  # 724 x 724 values are 4 MiB less 848 bytes
        A = torch.randn(n, m, generator=g, dtype=torch.float64)
        B = torch.randn(n, m, generator=g, dtype=torch.float64)
        ref = A.numpy().T @ B.numpy()
        out = ctx.project(A.cuda(), B.cuda())
        assert np.abs(out - ref).max() <= 1e-12 * np.abs(ref).max(), m
        Y = np.random.default_rng(m).standard_normal((m, m))
        Od = torch.zeros(n, m, dtype=torch.float64, device="cuda")
        ctx.combine(A.cuda(), Y, Od)
        ref = A.numpy() @ Y
        assert np.abs(Od.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max() * (m / 16), m


def test_solve_with_a_wide_subspace(fci10):
    """V^T HV of a wide subspace beyond the pinned memory that is kept."""
    cfg, ints, _ = fci10
    H = api.Hamiltonian(cfg, ints)
    H.build()
    ref = H.davidson(16, prec=api.FP64, tol=1e-5, graph=1)
    out = H.davidson(16, prec=api.FP64, tol=1e-5, max_subspace=17000, graph=1)  # 17000 x 32 values
    assert ref["converged"] and out["converged"]
    np.testing.assert_allclose(out["evals"], ref["evals"], rtol=0, atol=1e-8)
    again = H.davidson(16, prec=api.FP64, tol=1e-5, graph=1)
    assert np.array_equal(again["evals"], ref["evals"])
    H.close()
