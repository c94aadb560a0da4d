"""The compact string-driven products on the GPU: spaces whose blocks take
every grouping level (host counterpart: test_rascmp_host.py), at column
counts around every chunk width, against the oracle's stored sigma."""
import numpy as np
import pytest

import oracle
from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


def _mrci(ni, ne, nelec, m=2, ksym=1, seed=11):
    return (inputs.mrcisd_configs(ni, ne, nelec, max_external=m, ksym=ksym),
            inputs.make_integrals(ni + ne, seed, n_internal=ni))


SPACES = [
    ("level 1 and 2, 24-row groups cut at 8, 16 and 32 rows", lambda: _mrci(6, 8, 6)),
    ("no spin-flip symmetry", lambda: _mrci(6, 8, 6, ksym=2)),
    ("one external electron", lambda: _mrci(5, 9, 6, m=1)),
    ("two electrons", lambda: (inputs.fci_configs(5, 2), inputs.make_integrals(5, 9))),
    ("groups of one to 35 rows", lambda: (inputs.fci_configs(7, 8), inputs.make_integrals(7, 3))),
]


@pytest.mark.parametrize("name,make", SPACES, ids=[c[0] for c in SPACES])
def test_compact_products(name, make):
    cfg, ints = make()
    H = api.Hamiltonian(cfg, ints)
    assert H.direct_engine(2) == 2
    sp = oracle.OracleSpace(cfg, ints)
    sp.build_h()
    rng = np.random.default_rng(7)
    for k in (1, 2, 3, 4, 5, 8, 9, 16, 17, 19):
        X = rng.standard_normal((H.n, k))
        ref = sp.sigma(X)
        scale = np.abs(ref).max()
        y = H.sigma(X, api.DIRECT, api.FP64).reshape(ref.shape)
        assert np.abs(y - ref).max() <= 1e-12 * scale, k
        y32 = H.sigma(X.astype(np.float32), api.DIRECT, api.FP32).reshape(ref.shape)
        assert np.abs(y32 - ref).max() <= 2e-5 * scale, k
    H.close()
