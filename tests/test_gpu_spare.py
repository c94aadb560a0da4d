"""The scratch memory that a context keeps between calls: an allocation that
fails in one context gives back what the others keep, they work on without
it, and contexts of several threads may take and lose it at any time."""
import threading

import numpy as np
import pytest
import torch

from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


def _exhaust(H):
    """A solve whose basis cannot fit (568,204 x 568,204 values)."""
    with pytest.raises(api.PsociError) as e:
        H.davidson(1, prec=api.FP64, mode=api.DIRECT, max_subspace=H.n)
    assert e.value.code == api.ERR_NOMEM


@pytest.fixture(scope="module")
def large():
    cfg, ints, _ = inputs.workload("mrci8x24")
    H = api.Hamiltonian(cfg, ints)
    H.direct_engine()
    yield H
    H.close()


def test_other_contexts_give_back(fci10, large):
    cfg, ints, _ = fci10
    A = api.Hamiltonian(cfg, ints)
    A.build()
    h = A.get_h()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    _exhaust(large)
    assert torch.cuda.mem_get_info()[0] - before > 500 << 20
    A.build()
    for a, b in zip(A.get_h(), h):
        assert np.array_equal(a, b)
    A.close()


def test_threads_take_and_lose_scratch(large):
    cfg, ints = inputs.fci_configs(8, 6), inputs.make_integrals(8, 3)
    A = api.Hamiltonian(cfg, ints)
    A.build()
    h = A.get_h()
    ref = A.davidson(2, prec=api.FP64, tol=1e-8, want_vectors=False, graph=1)["evals"]
    A.close()
    errors = []

    def work():
        try:
            H = api.Hamiltonian(cfg, ints)
            for _ in range(8):
                H.set_integrals(ints)
                H.build()
                for a, b in zip(H.get_h(), h):
                    assert np.array_equal(a, b)
                e = H.davidson(2, prec=api.FP64, tol=1e-8, want_vectors=False, graph=1)["evals"]
                np.testing.assert_allclose(e, ref, rtol=0, atol=1e-9)
                H.rdm(np.ones(H.n))
            H.close()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for _ in range(8):
        _exhaust(large)
    for t in threads:
        t.join()
    assert not errors, errors[0]
