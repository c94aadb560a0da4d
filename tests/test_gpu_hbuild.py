"""The stored Hamiltonian on configuration lists whose blocks meet the edges
of the element batches (512) and steps (64): blocks of one element, blocks
longer than a batch, segments longer than a word, orbitals past the 32nd,
spin-orbit pairs; against the oracle's elements bit for bit, and its product
(which reads the transposed part too)."""
import numpy as np
import pytest

import oracle
from psoci_amd import api, inputs

pytestmark = pytest.mark.gpu


def _random(nbf, nelec, want, seed, open_max=10, jsym=(1,), high=0):
    """want distinct configurations near one reference (so that most connect)"""
    rng = np.random.default_rng(seed)
    base = np.zeros(nbf, np.int64)
    orbs = np.arange(nbf)[high:]
    for e in range(nelec):
        base[orbs[e % len(orbs)] if open_max > 8 else orbs[e // 2]] += 1
    seen = {}
    while len(seen) < want:
        o = base.copy()
        for _ in range(rng.integers(0, 4)):
            a, b = rng.choice(nbf, 2, replace=False)
            if o[a] > 0 and o[b] < 2:
                o[a] -= 1
                o[b] += 1
        if (o == 1).sum() <= open_max:
            seen.setdefault(tuple(o), len(seen))
    occ = np.array(list(seen), np.uint8)
    js = np.array([jsym[i % len(jsym)] for i in range(len(occ))], np.int32)
    return inputs.Configs(nbf, nelec, 1, occ, js)


def _closed(nbf, nelec, want):
    """closed shells only: blocks of one element"""
    rng = np.random.default_rng(8)
    seen = set()
    while len(seen) < want:
        o = np.zeros(nbf, np.uint8)
        o[rng.choice(nbf, nelec // 2, replace=False)] = 2
        seen.add(tuple(o))
    return inputs.Configs(nbf, nelec, 1, np.array(sorted(seen), np.uint8), np.ones(want, np.int32))


CASES = [
    ("one configuration", lambda: _random(4, 4, 1, 1)),
    ("blocks of one element", lambda: _closed(10, 8, 180)),
    ("10 open shells", lambda: _random(12, 10, 40, 2)),
    ("9 open shells", lambda: _random(11, 9, 40, 3)),
    ("45 orbitals", lambda: _random(45, 6, 300, 4, open_max=6, high=38)),
    ("odd, 40 orbitals", lambda: _random(40, 5, 200, 5, open_max=5, high=30)),
    ("spin-orbit", lambda: _random(9, 6, 150, 6, open_max=6, jsym=(1, 2, 3, 4))),
]


@pytest.mark.parametrize("name,make", CASES, ids=[c[0] for c in CASES])
def test_stored_matrix(name, make):
    cfg = make()
    sp = oracle.OracleSpace(cfg)
    H = api.Hamiltonian(cfg, inputs.make_integrals(cfg.nbf, 11))
    for seed in (11, 12):  # the second builds over the first
        ints = inputs.make_integrals(cfg.nbf, seed)
        sp.set_integrals(ints)
        H.set_integrals(ints)
        sp.build_h(8)
        assert H.build() == len(sp.val)
        rowptr, col, val, diag = H.get_h()
        np.testing.assert_array_equal(rowptr, sp.rowptr)
        np.testing.assert_array_equal(col, sp.col)
        assert np.array_equal(val, sp.val) and np.array_equal(diag, sp.diag)
        X = np.random.default_rng(seed).standard_normal((H.n, 4))
        ref = sp.sigma(X)
        y = H.sigma(X, api.STORED, api.FP64).reshape(ref.shape)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
    H.close()
