"""Tiles shared by several wavefronts: in systems with few tiles per class, each
wavefront takes a part of a tile's primitive quartets (bra primitives first, then
the ket's) and several blocks take one run.  Clusters from one water to six pass
through every number of wavefronts per tile, in FP64 and in mixed precision, with
pairs of 1 to 64 primitives (fewer than, equal to and not a multiple of the
shares).  FP64 is held to the 1e-10 of the unshared builds: partial sums only
reorder the additions, and each of the up to 64 partial contributions is rounded
to the accumulators' 2^-48.  Mixed precision is held to the path's 1e-6."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from quick_amd.basis import build_basis
from quick_amd.fock import FockEngine, QK_MIXED, make_opts
from quick_amd.geometry import synthetic_density, water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(1, 1, 1), (3, 1, 1), (3, 2, 1)], ids=lambda b: f"{b[0] * b[1] * b[2]}-waters")
def test_shared_tiles_against_oracle(box):
    print(f"[gpu-test] shared tiles {box}", flush=True)
    symbols, xyz = water_cluster(*box, seed=5)
    b = build_basis(symbols, np.asarray(xyz, float))
    D = synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, 3)
    eng = FockEngine(b)
    o = Oracle(b)
    o.set_cutoffs(*eng.compute_schwarz())
    Gref, nq, _ = o.fock(D, mode="cpu")
    gref, _, _ = o.grad(D)
    for opts, tol in ((make_opts(), 1e-10), (make_opts(precision=QK_MIXED, fp32_threshold=1e-3), 1e-6)):
        G = eng.fock(D, opts)
        assert eng.stats().quartets > 0
        assert np.array_equal(G, G.T)
        assert np.abs(G - Gref).max() <= tol
        assert np.abs(eng.grad(D, opts) - gref).max() <= tol
        # shares of a sum in fixed point: the same bits in any order
        assert np.array_equal(G, eng.fock(D, opts))
