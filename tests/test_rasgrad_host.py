"""The adjoint's matrices (ras_grad in psoci_amd/csrc/ras.cpp) on the host:
every block with pairs has the one of its sector, kind and budget, and blocks
without pairs (an orbital that every configuration fills) have none."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from psoci_amd import inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "psoci_amd", "csrc")
SRC = os.path.join(ROOT, "tests", "hostcheck", "host_rasgrad.cpp")
OUT = os.path.join(ROOT, "tests", "hostcheck", "_build", "libhostrasgrad.so")


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
    return ctypes.CDLL(OUT)


def _core(nbf, nelec, ksym=1):
    """Full CI with the first orbital doubly occupied throughout."""
    c = inputs.fci_configs(nbf, nelec, ksym=ksym)
    keep = c.occ[:, 0] == 2
    return inputs.Configs(nbf=nbf, nelec=nelec, ksym=ksym, occ=c.occ[keep].copy(), jsym=c.jsym[keep].copy())


# name, list, whether it has blocks without pairs
CASES = [
    ("fci 6/6", lambda: inputs.fci_configs(6, 6), False),
    ("fci 6/5", lambda: inputs.fci_configs(6, 5), False),
    ("mrcisd 4+5/4", lambda: inputs.mrcisd_configs(4, 5, 4), False),
    ("core 6/4", lambda: _core(6, 4), True),
    ("core 6/6", lambda: _core(6, 6), True),
    ("core 6/6 mult -1", lambda: _core(6, 6, ksym=2), True),
    ("core 6/5", lambda: _core(6, 5), True),
]


@pytest.mark.parametrize("name,make,empty", CASES, ids=[c[0] for c in CASES])
def test_adjoint_matrices(lib, name, make, empty):
    cfg = make()
    ints = inputs.make_integrals(cfg.nbf, 5)
    info = np.zeros(3, np.int64)
    arrays = [np.ascontiguousarray(cfg.occ, np.uint8), np.ascontiguousarray(cfg.jsym, np.int32), ints.valone,
              ints.valtwo, info]
    ptr = [a.ctypes.data_as(ctypes.c_void_p) for a in arrays]
    assert lib.hrg_check(cfg.nbf, cfg.nelec, cfg.ksym, ctypes.c_int64(cfg.ncfg), *ptr) == 0
    assert (info[1] > 0) == empty
    assert 0 < info[2] <= info[0] - info[1]


def test_limit_is_the_compact_layouts(lib):
    """The products' 31-bit offsets are those of the compact layout; the full
    one may be larger."""
    lim = 1 << 31
    for compact, full, limited in ((lim - 1, lim - 1, 0), (lim - 1, 2 * lim, 0), (lim, lim, 1), (lim, 2 * lim, 1)):
        assert lib.hrg_limited(ctypes.c_int64(compact), ctypes.c_int64(full)) == limited
