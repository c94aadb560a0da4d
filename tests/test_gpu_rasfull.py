"""One matrix per product: where the compact layouts' matrices (one per row
group) would take too much memory the plan keeps the full pair lists.  Sampled
rows of the sigma against the oracle's blocks on 42 million SEFs."""
from math import comb

import numpy as np
import pytest
import torch

import oracle
from psoci_amd import api, inputs
from test_gpu_direct import oracle_rows

pytestmark = pytest.mark.gpu


def _full_w(ni, ne, nelec):
    """W elements per column of the full pair lists, padded to 16, of an
    internal full CI with up to two electrons in the external orbitals."""
    def strings(n, c):
        return comb(ni, n - c) * comb(ne, c) if 0 <= c <= n else 0

    total = 0
    for dn in range(0, nelec + 1, 4):
        na, nb = (nelec + dn) // 2, (nelec - dn) // 2
        for kind, lu, lw in ((0, na - 1, nb - 1), (1, na - 2, nb), (2, na, nb - 2)):
            if min(lu, lw) < 0 or (kind == 2 and na == nb):
                continue
            for cu in range(3):
                for cw in range(3 - cu):
                    if kind == 0 and na == nb and cu > cw:
                        continue
                    u, w, b = strings(lu, cu), strings(lw, cw), 2 - cu - cw
                    rows = u * (u + 1) // 2 if kind == 0 and na == nb and cu == cw else u * w
                    if kind == 0:
                        q = ni * ni + (2 * ni * ne if b >= 1 else 0) + (ne * ne if b >= 2 else 0)
                    else:
                        q = comb(ni, 2) + (ni * ne if b >= 1 else 0) + (comb(ne, 2) if b >= 2 else 0)
                    total += rows * ((q + 15) // 16 * 16)
    return total


def test_one_matrix_per_product():
    if torch.cuda.mem_get_info()[0] < 270e9:
        pytest.skip("needs 270 GB of free device memory")
    cfg = inputs.mrcisd_configs(12, 24, 8)
    ints = inputs.make_integrals(36, 5, n_internal=12)
    H = api.Hamiltonian(cfg, ints)
    assert H.direct_engine(2) == 2
    assert H.direct_ras_info()["w_per_column"] == _full_w(12, 24, 8)
    sp = oracle.OracleSpace(cfg, ints)
    rng = np.random.default_rng(17)
    X = rng.standard_normal((H.n, 1))
    Y = H.sigma(X, api.DIRECT, api.FP64).reshape(X.shape)
    Y32 = H.sigma(X.astype(np.float32), api.DIRECT, api.FP32).reshape(X.shape)
    for I in [int(r) for r in rng.choice(cfg.ncfg, 4, replace=False)] + [0, cfg.ncfg - 1]:
        ref = oracle_rows(sp, cfg, I, X)
        rows = slice(int(sp.sef_off[I]), int(sp.sef_off[I]) + int(sp.nsef[I]))
        scale = max(1.0, np.abs(ref).max())
        assert np.abs(Y[rows] - ref).max() <= 1e-12 * scale, I
        assert np.abs(Y32[rows] - ref).max() <= 5e-5 * scale, I
    H.close()
