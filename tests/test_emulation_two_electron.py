"""The Fock and gradient kernels on the CPU, where an access
outside an allocation ends the process (tests/emulation): work lists, compacted
steps, pair records, prefetched kets and primitives, shared tiles and runs.

The systems pass through every form: one tile with 64 wavefronts on it (one
atom), several blocks per run, lists long enough to be compacted, with steps that
hold nothing (a cluster with the density of one molecule), exchange rows beyond LDS
(many functions), a gradient beyond LDS (many nuclei), pairs of 1 to 36
primitives; every class with d functions on one molecule, the others without.
Results against the oracle as on the device: FP64 1e-10, mixed 1e-6.
"""
import pytest

from tests import emulation

CODE = """
import sys
from tests.emulation import without_d
from tests.test_emulation import with_free_functions
from quick_amd.basis import build_basis
from quick_amd.geometry import synthetic_density, water_cluster
from oracle.oracle import Oracle
kind, tau, hybrid = ARGS
if kind[0] == "H":
    r = np.random.default_rng(3)
    sym, xyz = ["H"] * kind[1], 1.5 * r.uniform(size=(kind[1], 3))
else:
    sym, xyz = water_cluster(*kind[1], seed=5)
    xyz = np.asarray(xyz, float)
b = build_basis(list(sym), xyz)
if kind[0] != "d":
    b = without_d(b)
D = synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, 3)
if kind[0] == "masked":   # the density of one molecule: most kets fail the screen
    D[b.nbasis // 6:] = D[:, b.nbasis // 6:] = 0.0
if kind[0] == "free":
    b = with_free_functions(b, kind[2])
    full = np.zeros((b.nbasis, b.nbasis))
    full[kind[2]:, kind[2]:] = D
    D = full
if kind[0] == "nuclei":
    b.xyz = np.asfortranarray(np.concatenate([b.xyz, 9.0 + np.random.default_rng(4).uniform(size=(3, 2800))], axis=1))
e = FockEngine(b)
o = Oracle(b)
o.set_cutoffs(*e.compute_schwarz())
Gref, gref = o.fock(D, tau=tau, hybrid=hybrid, pair_cut=0.0, mode="gpu_cpuboys")[0], o.grad(D, cutoff=tau, hybrid=hybrid)[0]
for opts, tol in ((make_opts(tau=tau, hybrid=hybrid), 1e-10),
                  (make_opts(tau=tau, hybrid=hybrid, precision=QK_MIXED, fp32_threshold=1e-2), 1e-6)):
    G, g = e.fock(D, opts), e.grad(D, opts)
    assert np.abs(G - Gref).max() <= tol and np.abs(g - gref).max() <= tol, (np.abs(G - Gref).max(), np.abs(g - gref).max())
    if kind[0] == "free":
        continue   # beyond the no-allocation entry's scratch
    Df, G2 = np.asfortranarray(D).ravel(order="F").copy(), np.zeros(b.nbasis ** 2)
    assert e.fock_device_noalloc(Df.ctypes.data, G2.ctypes.data, opts) == 0   # the lists without compaction
    assert np.array_equal(G2, G.ravel(order="F"))
print(emu.emu_record().decode())
"""

TAU = 1e-11
CASES = {"1-atom": (("H", 1), TAU, 1.0), "2-atoms": (("H", 2), 1e-6, 0.0), "5-atoms": (("H", 5), TAU, 0.2),
         "3-waters": (("water", (3, 1, 1)), TAU, 1.0),
         "6-waters": (("water", (3, 2, 1)), TAU, 1.0), "masked": (("masked", (3, 2, 1)), TAU, 1.0),
         "d": (("d", (1, 1, 1)), TAU, 1.0), "functions": (("free", (1, 1, 1), 3300), TAU, 1.0), "nuclei": (("nuclei", (1, 1, 1)), TAU, 1.0)}


@pytest.mark.parametrize("name,low", [(n, low) for n in CASES for low in (False, True)
                                      if not (low and n in ("3-waters", "6-waters", "functions", "nuclei"))],
                         ids=lambda v: v if isinstance(v, str) else ("low" if v else "high"))
def test_two_electron_kernels_stay_in_bounds(emulated_lib, name, low):
    record = emulation.run(emulated_lib, CODE.replace("ARGS", repr(CASES[name])), low=low)
    launched = [line.split() for line in record.splitlines() if line]
    modes = {(n.split("ELi")[-1][0], "f32" in n) for n, *_ in launched if "fock_kernel" in n}
    compacted = any("compact_kernel" in n for n, *_ in launched)
    # the forms this case is here for
    if name in ("6-waters", "masked"):
        assert compacted
    if name == "functions":
        assert {("0", False), ("0", True)} <= modes
    if name == "1-atom":
        assert max(int(g) for n, g, *_ in launched if "fock_kernel" in n) >= 4
