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
def test_functions_outside_every_shell(emulated_lib, k, low):
    """lanes without a shell pair read nothing of the functions that no shell holds; tolerances as on the device"""
    out = emulation.run(emulated_lib, f"from tests.test_emulation import *\nprint(*free_function_errors({k}))", low=low)
    dS, dH, free, dg = map(float, out.split())
    assert dS <= 1e-12 and dH <= 1e-10 and free == 0.0 and dg <= 1e-10


def odd_shells(kind):
    """(tables for the library, basis for the oracle) of two waters with shells that do not hold each Cartesian
    component of their angular momentum once"""
    s, x = water_cluster(2, 1, 1, seed=5)
    b = build_basis(s, np.asarray(x, float))
    b.KLMN = b.KLMN.copy()
    f0 = lambda sh, L: int(b.ksumtype[sh]) - 1 + int(b.Qsbasis[sh, L])
    sp = next(i for i in range(b.nshell) if b.Qfinal[i] == 1)
    d = next(i for i in range(b.nshell) if b.Qfinal[i] == 2)
    if kind == "twice":        # p functions x, x, z
        b.KLMN[:, f0(sp, 1) + 1] = b.KLMN[:, f0(sp, 1)]
    elif kind == "other-l":    # a p function among the d, an s among the p, a p in an s shell
        b.KLMN[:, f0(d, 2) + 3] = (0, 1, 0)
        b.KLMN[:, f0(sp, 1) + 2] = 0
    elif kind == "order":      # a permuted d shell stays whole
        n = np.arange(f0(d, 2), f0(d, 2) + 6)
        b.KLMN[:, n] = b.KLMN[:, n[[3, 5, 0, 4, 1, 2]]]
    if kind != "shared":
        return b, b
    # a hydrogen's second s shell (one primitive) claims the function of its first (three)
    h = next(i for i in range(b.nshell) if b.kprim[i] == 3 and b.Qfinal[i] == 0)
    f = f0(h, 0)
    c, o = copy.copy(b), copy.copy(b)
    c.ksumtype = np.array(b.ksumtype)
    c.ksumtype[h + 1] = c.ksumtype[h]
    o.ncontract, o.dcoeff, o.aexp = b.ncontract.copy(), b.dcoeff.copy(), b.aexp.copy()
    o.ncontract[f] = 1
    o.dcoeff[:, f] = b.gccoeff[:, f] * b.cons[f]
    o.aexp[:, f] = b.gcexpo[:, f]
    o.ncontract[f + 1] = 0     # held by no shell now
    return c, o


def odd_shell_errors(kind):
    """one-electron integrals and gradient of such a basis against the oracle's, which go function by function"""
    from oracle import oracle as O
    from quick_amd.fock import FockEngine
    lib, ref = odd_shells(kind)
    e = FockEngine(lib)
    e.set_charges(ref.Z.astype(float))
    S, H = e.oneint()
    So, Ho = O.hcore(ref)
    D, W = (synthetic_density(ref.xyz, ref.katom, ref.ksumtype, ref.nbasis, q) for q in (3, 4))
    return np.abs(S - So).max(), np.abs(H - Ho).max(), np.abs(e.oneint_grad(D, W) - O.oneint_grad(ref, D, W)).max()


ODD = ["twice", "other-l", "order", "shared"]


@pytest.mark.parametrize("kind", ODD)
def test_shells_without_each_component_once(emulated_lib, kind):
    out = emulation.run(emulated_lib, f"from tests.test_emulation import *\nprint(*odd_shell_errors({kind!r}))")
    dS, dH, dg = map(float, out.split())
    assert dS <= 1e-12 and dH <= 1e-10 and dg <= 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ODD)
def test_shells_without_each_component_once_on_the_device(kind):
    print(f"[gpu-test] odd shells: {kind}", flush=True)
    dS, dH, dg = odd_shell_errors(kind)
    assert dS <= 1e-12 and dH <= 1e-10 and dg <= 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 6])
def test_functions_outside_every_shell_on_the_device(k):
    print(f"[gpu-test] {k} functions outside every shell", flush=True)
    dS, dH, free, dg = free_function_errors(k)
    assert dS <= 1e-12 and dH <= 1e-10 and free == 0.0 and dg <= 1e-10


JOIN = """
from tests.emulation import without_d
from quick_amd.basis import build_basis
from quick_amd.geometry import synthetic_density
b = without_d(build_basis(["H", "H"], np.array([[0.0, 0.0, 0.0], [0.3, 0.5, 0.7]])))
D = synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, 3).ravel(order="F").copy()
W = D.copy()
e = FockEngine(b)
e.compute_schwarz()
e.set_charges([1.0, 1.0])
emu.emu_fail_in.argtypes = [C.c_longlong]
o = make_opts(**KW)
e.prepare(o)
p = lambda a: C.c_void_p(a.ctypes.data)
calls = {"fock": lambda x: lib().qk_fock_device(e.h, p(D), p(x), C.byref(o), None),
         "grad": lambda x: lib().qk_grad_device(e.h, p(D), p(x), C.byref(o), None),
         "oneint": lambda x: lib().qk_oneint_device(e.h, p(x), None, None),
         "oneint_grad": lambda x: lib().qk_oneint_grad_device(e.h, p(D), p(W), p(x), None)}
for name, call in calls.items():
    new = lambda: np.zeros(3 * b.natom if "grad" in name else b.nbasis ** 2)
    good = new()
    assert call(good) == 0 and emu.emu_unjoined() == 0, name
    failed = 0
    for n in range(1000):
        emu.emu_fail_in(n)
        rc = call(new())
        emu.emu_fail_in(-1)
        assert emu.emu_unjoined() == 0, f"{name}: error {n} leaves {emu.emu_unjoined()} streams forked"
        if rc == 0:
            break
        failed += 1
        again = new()
        assert call(again) == 0 and np.array_equal(again, good), f"{name} after error {n}"
    print(name, failed)
"""


@pytest.mark.parametrize("kw", ["dict()", "dict(precision=QK_MIXED, fp32_threshold=1e-1)"], ids=["fp64", "mixed"])
def test_streams_are_joined_after_any_error(emulated_lib, kw):
    """every launch check of a call fails once: the call reports it, the streams it forked are ordered before what
    follows on the caller's, and the next call gives the same result as before"""
    out = dict(line.split() for line in emulation.run(emulated_lib, JOIN.replace("KW", kw)).splitlines())
    assert int(out["fock"]) >= 8 and int(out["grad"]) >= 8 and int(out["oneint"]) and int(out["oneint_grad"]), out


SCRATCH = """
from tests.emulation import without_d
from quick_amd.basis import build_basis
from quick_amd.geometry import synthetic_density, water_cluster
emu.emu_set_scratch.argtypes = [C.c_char_p, C.c_longlong]
for name in NAMES:
    emu.emu_set_scratch(name.encode(), 1 << 20)
def both(b):
    D = synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, 3)
    e = FockEngine(b)
    e.set_charges(b.Z.astype(float))
    return e, D
s, x = water_cluster(3, 2, 1, seed=2)
e, D = both(build_basis(s, np.asarray(x, float)))
e.oneint_grad(D, D)
e, D = both(without_d(build_basis(["H"] * 3, np.array([[0.0, 0.0, 0.0], [0.3, 0.5, 0.7], [1.1, 0.2, 0.4]]))))
e.compute_schwarz()
for o in (make_opts(), make_opts(precision=QK_MIXED, fp32_threshold=1e-1)):
    e.fock(D, o), e.grad(D, o)
print(emu.emu_record().decode())
"""


def test_grids_of_spilling_kernels(emulated_lib):
    """the grids that the launchers really use, were every kernel that can spill to take 1 MiB per lane (the budget
    then holds one block of 256 threads): no launch may back more than the budget"""
    names = ["oneint_grad_kernel", "grad_light_kernel", "fock_kernel"]
    nm = emulation.symbols(emulated_lib)
    spill = [n for n in nm if any(k in n for k in names) and "launch" not in n]
    assert len(spill) >= 6 + 12 + 12
    seen = set()
    for line in emulation.run(emulated_lib, SCRATCH.replace("NAMES", repr(spill))).split("\n"):
        if line:
            name, grid, block, _, _ = line.split()
            if name in spill:
                seen.add(name)
                assert int(grid) == 1 and int(block) == 256, line
    assert len(seen) >= 6 + 6 + 6


def far_charge_errors():
    """a hydrogen molecule and a bare charge 1e25 bohr away, against the oracle: |dH|, |d one-electron grad|"""
    from oracle import oracle as O
    from quick_amd.fock import FockEngine
    b = build_basis(["H", "H"], np.array([[0.0, 0.0, 0.0], [0.3, 0.5, 0.7]]))
    b.xyz = np.asfortranarray(np.concatenate([b.xyz, [[1e25], [0.0], [0.0]]], axis=1))
    b.Z = np.array([1, 1, 1])
    D, W = (synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, q) for q in (3, 4))
    e = FockEngine(b)
    e.set_charges(b.Z.astype(float))
    return np.abs(e.oneint()[1] - O.hcore(b)[1]).max(), np.abs(e.oneint_grad(D, W) - O.oneint_grad(b, D, W)).max()


def test_charge_very_far_away(emulated_lib):
    """Boys arguments of 1e50, beyond what exp's reduction can carry: finite, as the oracle has them"""
    out = emulation.run(emulated_lib, "from tests.test_emulation import *\nprint(*far_charge_errors())")
    assert all(float(v) <= 1e-10 for v in out.split()), out


@pytest.mark.gpu
def test_charge_very_far_away_on_the_device():
    print("[gpu-test] a charge very far away", flush=True)
    assert all(v <= 1e-10 for v in far_charge_errors())


TIMING = """
from tests.emulation import without_d
from quick_amd.basis import build_basis
from quick_amd.geometry import synthetic_density
b = without_d(build_basis(["H", "H"], np.array([[0.0, 0.0, 0.0], [0.3, 0.5, 0.7]])))
D = synthetic_density(b.xyz, b.katom, b.ksumtype, b.nbasis, 3)
e = FockEngine(b)
e.compute_schwarz()
for on in (False, True):
    e.set_timing(on)
    for o in (make_opts(), make_opts(precision=QK_MIXED, fp32_threshold=1e-1)):
        for call in (e.fock, e.grad):
            call(D, o)   # the lists
            emu.emu_clear_record()
            call(D, o)
            print(on, *{line.split()[-1] for line in emu.emu_record().decode().splitlines()})
"""


def test_timed_classes_run_alone(emulated_lib):
    """per-class times are those of one kernel at a time: with timing on, a call works on the caller's stream only"""
    for line in emulation.run(emulated_lib, TIMING).splitlines():
        on, *streams = line.split()
        assert (streams == ["0"]) == (on == "True"), line
