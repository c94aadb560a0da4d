"""FP64 solves whose blocks stay orthonormal through two fused Gram-Schmidt
passes or fall back to the separate ones: blocks as large as the space's
basis allows, starting vectors that are nearly the solutions (corrections
almost within the basis), residuals to 1e-10."""
import numpy as np
import pytest

import oracle
from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbf,nelec,k", [(3, 4, 2), (5, 4, 12), (6, 6, 8), (7, 4, 1)])
@pytest.mark.parametrize("precond", [0, 1])
def test_vectors_orthonormal(nbf, nelec, k, precond):
    cfg = inputs.fci_configs(nbf, nelec)
    ints = inputs.make_integrals(nbf, 31 + nbf)
    sp = oracle.OracleSpace(cfg, ints)
    sp.build_h(8)
    A = sp.dense_h()
    w, U = np.linalg.eigh(A)
    H = api.Hamiltonian(cfg, ints)
    rng = np.random.default_rng(k)
    near = np.linalg.qr(U[:, :k] + 1e-7 * rng.standard_normal((H.n, k)))[0]
    for kw in (dict(guess=0), dict(guess=1), dict(guess=2, guess_vectors=np.ascontiguousarray(near))):
        out = H.davidson(k, prec=api.FP64, mode=api.DIRECT, tol=1e-10, precond=precond, **kw)
        assert out["converged"]
        # converged pairs are eigenpairs (which of two degenerate roots the
        # unit vectors reach is not promised); eigenvalue errors are the
        # squares of the residuals; vectors orthonormal to a few hundred
        # roundings
        E = np.asarray(out["evals"])
        assert np.abs(w[:, None] - E).min(axis=0).max() <= 1e-11 and (np.diff(E) >= -1e-11).all()
        assert abs(E[0] - w[0]) <= 1e-11
        V = np.asarray(out["evecs"]).reshape(H.n, k)
        assert np.linalg.norm(A @ V - V * E, axis=0).max() <= 2e-10
        assert np.abs(V.T @ V - np.eye(k)).max() <= 1e-13
    H.close()
