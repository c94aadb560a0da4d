"""The stored sigma at every kernel width and shape, on spaces whose rows end
inside a turn of every lane count, against the product with the exported
matrix (scipy, FP64)."""
import numpy as np
import pytest
import scipy.sparse as sp

from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu

SPACES = [
    ("2 rows", lambda: (inputs.fci_configs(2, 2), inputs.make_integrals(2, 3))),
    ("fci 5/4", lambda: (inputs.fci_configs(5, 4), inputs.make_integrals(5, 4))),
    ("fci 6/5", lambda: (inputs.fci_configs(6, 5), inputs.make_integrals(6, 6))),
    ("17,000 rows", lambda: (inputs.mrcisd_configs(6, 8, 6), inputs.make_integrals(14, 7, n_internal=6))),
]


@pytest.mark.parametrize("shape", [None, "1x8", "2x2", "4x4", "4x1"])
@pytest.mark.parametrize("name,make", SPACES, ids=[c[0] for c in SPACES])
def test_stored_sigma_widths(name, make, shape, monkeypatch):
    if shape:
        monkeypatch.setenv("PSOCI_SPMM_SHAPE", shape)
    cfg, ints = make()
    H = api.Hamiltonian(cfg, ints)
    H.build()
    rowptr, col, val, diag = H.get_h()
    L = sp.csr_matrix((val, col, rowptr), shape=(H.n, H.n))
    A = L + L.T - sp.diags(diag)
    rng = np.random.default_rng(3)
    for k in (1, 2, 3, 4, 7, 8, 16, 20, 32, 35):
        X = rng.standard_normal((H.n, k))
        ref = A @ X
        scale = np.abs(ref).max()
        y = H.sigma(X, api.STORED, api.FP64).reshape(ref.shape)
        assert np.abs(y - ref).max() <= 1e-12 * scale, k
        y32 = H.sigma(X.astype(np.float32), api.STORED, api.FP32).reshape(ref.shape)
        assert np.abs(y32 - ref).max() <= 2e-5 * scale, k
    H.close()


RULE = [
    # rows per wavefront of 16 columns, FP64 and FP32, by the number of rows
    ("2,044 rows", lambda: (inputs.fci_configs(8, 6), inputs.make_integrals(8, 4)), 1, 1),
    ("18,354 rows", SPACES[3][1], 2, 2),
    ("31,650 rows", lambda: (inputs.fci_configs(10, 8), inputs.make_integrals(10, 4)), 8, 4),
]


@pytest.mark.parametrize("name,make,r64,r32", RULE, ids=[c[0] for c in RULE])
def test_rows_per_wavefront(name, make, r64, r32):
    """Whole rounds of workgroups over 256 compute units."""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("another number of compute units")
    cfg, ints = make()
    H = api.Hamiltonian(cfg, ints)
    H.build()
    assert H.stored_shape(api.FP64)["rows_per_wave"] == r64
    assert H.stored_shape(api.FP32)["rows_per_wave"] == r32
    H.close()
