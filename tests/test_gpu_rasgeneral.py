"""The automatic choice's string plans of lists that are part of a space and
of odd electron counts: against the configuration engine (sigma, adjoint,
Davidson roots); requests for engine 2 stay refused, small lists stay on the
configuration records."""
import numpy as np
import pytest

from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


def _part(cfg, share, seed=9):
    keep = np.random.default_rng(seed).random(cfg.ncfg) < share
    return inputs.Configs(nbf=cfg.nbf, nelec=cfg.nelec, ksym=cfg.ksym, occ=cfg.occ[keep].copy(),
                          jsym=cfg.jsym[keep].copy())


def _ints(ni, ne):
    return inputs.make_integrals(ni + ne, 21, n_internal=ni)


SPACES = [
    ("part of mrcisd 8+14/6", lambda: (_part(inputs.mrcisd_configs(8, 14, 6), 0.7), _ints(8, 14))),
    ("part of mrcisd 8+14/6, mult -1", lambda: (_part(inputs.mrcisd_configs(8, 14, 6, ksym=2), 0.7), _ints(8, 14))),
    ("odd mrcisd 7+14/5", lambda: (inputs.mrcisd_configs(7, 14, 5), _ints(7, 14))),
    ("odd mrcisd 7+10/7, alpha and beta swapped",
     lambda: (inputs.mrcisd_configs(7, 10, 7, jsym=3, ksym=3), _ints(7, 10))),
]


@pytest.mark.parametrize("name,make", SPACES, ids=[c[0] for c in SPACES])
def test_general_plan_matches_records(name, make):
    cfg, ints = make()
    A = api.Hamiltonian(cfg, ints)
    assert A.direct_engine(1) == 1
    B = api.Hamiltonian(cfg, ints)
    assert B.direct_engine() == 2
    with pytest.raises(api.PsociError) as e:
        B.direct_engine(2)
    assert e.value.code == api.ERR_UNSUPPORTED
    assert B.direct_engine() == 2
    rng = np.random.default_rng(2)
    for k in (1, 3, 8, 16, 18):  # widths change between calls: the absent determinants stay zero
        X = rng.standard_normal((A.n, k))
        ya = A.sigma(X, api.DIRECT, api.FP64)
        scale = np.abs(ya).max()
        assert np.abs(B.sigma(X, api.DIRECT, api.FP64) - ya).max() <= 1e-12 * scale, k
        y32 = B.sigma(X.astype(np.float32), api.DIRECT, api.FP32)
        assert np.abs(y32 - ya).max() <= 2e-5 * scale, k
    C = rng.standard_normal((A.n, 3)) / np.sqrt(A.n)
    w = np.array([1.0, -0.4, 0.3])
    a1, a2, _ = A.rdm(C, w)
    b1, b2, _ = B.rdm(C, w)
    scale = max(np.abs(a1).max(), np.abs(a2).max())
    assert np.abs(b1 - a1).max() <= 1e-12 * scale
    assert np.abs(b2 - a2).max() <= 1e-12 * scale
    a = A.davidson(2, prec=api.MIXED, mode=api.DIRECT, tol=1e-6, want_vectors=False)
    b = B.davidson(2, prec=api.MIXED, mode=api.DIRECT, tol=1e-6, want_vectors=False)
    assert a["converged"] and b["converged"]
    np.testing.assert_allclose(b["evals"], a["evals"], atol=1e-9, rtol=0)
    A.close()
    B.close()


def test_small_or_thin_lists_stay_on_the_records():
    for cfg, ints in ((_part(inputs.mrcisd_configs(8, 14, 6), 0.05), _ints(8, 14)),
                      (inputs.mrcisd_configs(4, 4, 5), _ints(4, 4))):
        H = api.Hamiltonian(cfg, ints)
        assert H.direct_engine() == 1
        with pytest.raises(api.PsociError):
            H.direct_engine(2)
        assert H.direct_engine() == 1
        H.close()


@pytest.mark.parametrize("fails", ["sigma", "rdm"])
def test_unmet_request_is_forgotten(fails):
    """A request for engine 2 that a call finds impossible does not keep the
    automatic choice, asked for again, from the strings."""
    cfg, ints = SPACES[2][1]()
    H = api.Hamiltonian(cfg, ints)
    X = np.random.default_rng(2).standard_normal((H.n, 2))
    assert H.direct_engine(2, build=False) is None
    if fails == "sigma":
        with pytest.raises(api.PsociError) as e:
            H.sigma(X, api.DIRECT)
        assert e.value.code == api.ERR_UNSUPPORTED
    else:
        H.rdm(X)  # the pair walk
    H.direct_engine(0, build=False)
    assert H.direct_engine() == 2
    H.close()
