"""The compact layout of the string-driven products (RasCmp in
psoci_amd/csrc/ras.hpp) on the host: rows and pairs invert, groups cover the
rows, and the sigma through the compact matrices equals the oracle's."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle
from psoci_amd import inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "psoci_amd", "csrc")
SRC = os.path.join(ROOT, "tests", "hostcheck", "host_rascmp.cpp")
OUT = os.path.join(ROOT, "tests", "hostcheck", "_build", "libhostrascmp.so")


@pytest.fixture(scope="module")
def lib():
    deps = [SRC] + [os.path.join(CSRC, f) for f in ("ras.cpp", "ras.hpp", "space.cpp", "elem.hpp", "common.hpp")]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(d) for d in deps):
        os.makedirs(os.path.dirname(OUT), exist_ok=True)
        if not os.path.exists("/opt/rocm/bin/hipcc"):
            pytest.skip("hipcc not available")
        subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared",
                        "-ffp-contract=off", "-x", "hip", SRC, os.path.join(CSRC, "space.cpp"),
                        os.path.join(CSRC, "ras.cpp"), "-o", OUT], check=True)
    L = ctypes.CDLL(OUT)
    P = ctypes.c_void_p
    L.hrc_sigma.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int64, P, P, P, P, ctypes.c_int, P, P,
                            P, ctypes.c_int]
    return L


def _fci(nbf, nelec, ksym=1):
    return inputs.fci_configs(nbf, nelec, ksym=ksym), inputs.make_integrals(nbf, 5)


def _mrci(ni, ne, nelec, m=2, ksym=1):
    return (inputs.mrcisd_configs(ni, ne, nelec, max_external=m, ksym=ksym),
            inputs.make_integrals(ni + ne, 11, n_internal=ni))


def _moved(cfg, ints, seed=3):
    """The same kind of space with the external orbitals spread among the internal ones."""
    perm = np.random.default_rng(seed).permutation(cfg.nbf)
    return (inputs.Configs(nbf=cfg.nbf, nelec=cfg.nelec, ksym=cfg.ksym, occ=cfg.occ[:, perm].copy(), jsym=cfg.jsym),
            ints)


# name, space, levels that must occur
CASES = [
    ("fci 6/6", lambda: _fci(6, 6), (1,)),
    ("fci 6/6 mult -1", lambda: _fci(6, 6, ksym=2), (1,)),
    ("fci 8/8", lambda: _fci(8, 8), (1,)),
    ("fci 7/2", lambda: _fci(7, 2), (0,)),
    ("mrcisd 4+5/4", lambda: _mrci(4, 5, 4), (1,)),
    ("mrcisd 3+9/4", lambda: _mrci(3, 9, 4), ()),
    ("mrcisd 3+9/4 mult -1", lambda: _mrci(3, 9, 4, ksym=2), ()),
    ("mrcisd 3+4/6", lambda: _mrci(3, 4, 6), (0,)),
    ("mrcis 4+8/4", lambda: _mrci(4, 8, 4, m=1), ()),
    ("mrcisd 4+8/4, orbitals interleaved", lambda: _moved(*_mrci(4, 8, 4)), (1,)),
    ("mrcisd 2+8/6", lambda: _mrci(2, 8, 6), ()),
    ("mrcisd 6+8/6", lambda: _mrci(6, 8, 6), (1, 2)),
    ("mrcisd 6+8/6 mult -1", lambda: _mrci(6, 8, 6, ksym=2), (1, 2)),
]


def _run(lib, cfg, ints, general):
    sp = oracle.OracleSpace(cfg, ints)
    sp.build_h()
    X = np.random.default_rng(3).standard_normal((sp.n, 2))
    ref = sp.sigma(X)
    Y = np.zeros_like(X)
    info = np.zeros(6)
    occ = np.ascontiguousarray(cfg.occ, np.uint8)
    js = np.ascontiguousarray(cfg.jsym, np.int32)
    ptr = [a.ctypes.data_as(ctypes.c_void_p) for a in (occ, js, ints.valone, ints.valtwo)]
    rc = lib.hrc_sigma(cfg.nbf, cfg.nelec, cfg.ksym, cfg.ncfg, *ptr, X.shape[1],
                       X.ctypes.data_as(ctypes.c_void_p), Y.ctypes.data_as(ctypes.c_void_p),
                       info.ctypes.data_as(ctypes.c_void_p), general)
    return rc, Y, ref, info


@pytest.mark.parametrize("name,make,levels", CASES, ids=[c[0] for c in CASES])
def test_compact_products_match_oracle(lib, name, make, levels):
    rc, Y, ref, info = _run(lib, *make(), 0)
    assert rc == 0, rc
    np.testing.assert_allclose(Y, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    for lev in levels:
        assert info[lev] > 0, info
    assert info[4] <= info[3]
    assert info[5] == 1.0


@pytest.mark.parametrize("name,make,levels", [c for c in CASES if c[2]], ids=[c[0] for c in CASES if c[2]])
def test_layouts_without_dropped_pairs(lib, name, make, levels):
    rc, Y, ref, info = _run(lib, *make(), 2)
    assert rc == 0, rc
    np.testing.assert_allclose(Y, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    assert info[1] == info[2] == 0 and info[4] == info[3]


def _part(cfg, ints, share, seed=9):
    keep = np.random.default_rng(seed).random(cfg.ncfg) < share
    return (inputs.Configs(nbf=cfg.nbf, nelec=cfg.nelec, ksym=cfg.ksym, occ=cfg.occ[keep].copy(),
                           jsym=cfg.jsym[keep].copy()), ints)


def _odd(cfg, ints, jsym):
    return inputs.Configs(nbf=cfg.nbf, nelec=cfg.nelec, ksym=jsym, occ=cfg.occ,
                          jsym=np.full(cfg.ncfg, jsym, np.int32)), ints


GENERAL = [
    ("part of fci 6/6", lambda: _part(*_fci(6, 6), 0.5)),
    ("part of fci 6/6, mult -1", lambda: _part(*_fci(6, 6, ksym=2), 0.5)),
    ("part of mrcisd 5+5/4", lambda: _part(*_mrci(5, 5, 4), 0.3)),
    ("odd fci 6/5", lambda: _fci(6, 5)),
    ("odd fci 6/7, alpha and beta swapped", lambda: _odd(*_fci(6, 7), 3)),
    ("odd mrcisd 4+5/5", lambda: _mrci(4, 5, 5)),
    ("odd mrcisd 6+8/5", lambda: _mrci(6, 8, 5)),
    ("part of odd mrcisd 4+5/3", lambda: _part(*_mrci(4, 5, 3), 0.6)),
]


@pytest.mark.parametrize("name,make", GENERAL, ids=[c[0] for c in GENERAL])
def test_general_plans_match_oracle(lib, name, make):
    """Lists that are part of a space, and odd electron counts: refused
    without `general`, the oracle's sigma with it."""
    cfg, ints = make()
    rc, _, _, _ = _run(lib, cfg, ints, 0)
    assert rc == 1
    rc, Y, ref, info = _run(lib, cfg, ints, 1)
    assert rc == 0, rc
    assert (info[5] < 1.0) == name.startswith("part")
    np.testing.assert_allclose(Y, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
