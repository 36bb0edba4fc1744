"""One-electron kernels where their work split has its edges: a single shell pair,
every bucket of primitive pairs (1 to 64), wavefronts that are not full, and more
than one row of blocks over the nuclei (from 16 nuclei on; the last row uneven).
The random density is not the wave function's, so every element counts.  Against
the oracle's restatement: S to 1e-12 and H to 1e-10 as in the other one-electron
tests, the gradient to 1e-10 per nucleus (its terms are below 1e3 and their FP64
sums differ in order only)."""
import numpy as np
import pytest

from oracle import oracle as O
from quick_amd.basis import build_basis
from quick_amd.fock import FockEngine
from quick_amd.geometry import synthetic_density, water_cluster

pytestmark = pytest.mark.gpu
ZOF = {"H": 1.0, "O": 8.0}
CASES = {"H": (["H"], [[0.0, 0.0, 0.0]]), "O-H": (["O", "H"], [[0.0, 0.0, 0.0], [0.3, 0.5, 0.7]]),
         "15-atoms": water_cluster(5, 1, 1, seed=2), "18-atoms": water_cluster(3, 2, 1, seed=2),
         "27-atoms": water_cluster(3, 3, 1, seed=2)}


@pytest.mark.parametrize("name", CASES)
def test_oneint_edges(name):
    print(f"[gpu-test] one-electron edges {name}", flush=True)
    symbols, xyz = CASES[name]
    b = build_basis(symbols, np.asarray(xyz, float))
    eng = FockEngine(b)
    eng.set_charges([ZOF[s] for s in symbols])
    S, H = eng.oneint()
    So, Ho = O.hcore(b)
    assert np.abs(S - So).max() <= 1e-12 and np.abs(H - Ho).max() <= 1e-10
    assert np.array_equal(S, S.T) and np.array_equal(H, H.T)
    D, W = (synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, s) for s in (3, 4))
    g = eng.oneint_grad(D, W)
    assert np.abs(g - O.oneint_grad(b, D, W)).max() <= 1e-10
    assert np.array_equal(g, eng.oneint_grad(D, W))
