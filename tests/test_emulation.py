"""The device code on the CPU (tests/emulation), where an access outside a device
allocation or a block's LDS ends the process: each allocation lies against an
inaccessible page, once at its end (high) and once at its start (low)."""
import copy

import numpy as np
import pytest

from tests import emulation
from quick_amd.basis import build_basis
from quick_amd.geometry import synthetic_density, water_cluster

ZOF = {"H": 1.0, "O": 8.0}


@pytest.fixture(scope="session")
def lib(tmp_path_factory):
    return emulation.build(tmp_path_factory.mktemp("emulation"))


def with_free_functions(b, k):
    """the basis with k functions in front that belong to no shell"""
    c = copy.copy(b)
    c.nbasis, c.ksumtype, c.cons = b.nbasis + k, np.asarray(b.ksumtype) + k, np.concatenate([np.ones(k), b.cons])
    for f in ("KLMN", "gccoeff", "gcexpo"):
        a = np.asarray(getattr(b, f))
        setattr(c, f, np.concatenate([np.zeros((a.shape[0], k), a.dtype), a], axis=1))
    return c


def free_function_errors(k):
    """one-electron integrals and gradient with k functions outside every shell, whose density is NaN, against the
    oracle's for the others: max |dS|, |dH|, the free functions' largest element, max |dgrad|"""
    from oracle import oracle as O
    from quick_amd.fock import FockEngine
    s, x = water_cluster(2, 1, 1, seed=5)
    b = build_basis(s, np.asarray(x, float))
    c = with_free_functions(b, k)
    e = FockEngine(c)
    e.set_charges([ZOF[t] for t in s])
    S, H = e.oneint()
    So, Ho = O.hcore(b)
    D, W = (synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, q) for q in (3, 4))
    nan = [np.full((c.nbasis, c.nbasis), np.nan) for _ in (D, W)]
    for full, part in zip(nan, (D, W)):
        full[k:, k:] = part
    g = e.oneint_grad(*nan)
    return (np.abs(S[k:, k:] - So).max(), np.abs(H[k:, k:] - Ho).max(), max(np.abs(S[:k]).max(), np.abs(H[:k]).max()),
            np.abs(g - O.oneint_grad(b, D, W)).max())


@pytest.mark.parametrize("low", [False, True], ids=["high", "low"])
@pytest.mark.parametrize("k", [1, 6])
def test_functions_outside_every_shell(lib, k, low):
    """lanes without a shell pair read nothing of the functions that no shell holds; tolerances as on the device"""
    out = emulation.run(lib, f"from tests.test_emulation import *\nprint(*free_function_errors({k}))", low=low)
    dS, dH, free, dg = map(float, out.split())
    assert dS <= 1e-12 and dH <= 1e-10 and free == 0.0 and dg <= 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 6])
def test_functions_outside_every_shell_on_the_device(k):
    print(f"[gpu-test] {k} functions outside every shell", flush=True)
    dS, dH, free, dg = free_function_errors(k)
    assert dS <= 1e-12 and dH <= 1e-10 and free == 0.0 and dg <= 1e-10
