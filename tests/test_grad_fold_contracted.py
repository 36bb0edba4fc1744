"""The density-folded gradient code on contracted shells: three primitives for
every s and p function and two for every d, so that the sums over primitive
quartets which meet the density after the loop (S) hold 16 to 81 terms in every
class.

Everything is linear in the primitive quartets, so the error of a contracted
sum is bounded by the sum of theirs: it is held to 1e-11 (FP64) and 2e-5 (FP32),
the fractions that tests/test_grad_fold.py takes for a single quartet, of the sum
over the primitive quartets of each one's largest derivative.
"""
import ctypes
import math

import numpy as np
import pytest

from oracle.oracle import fmt
from tests.test_grad_fold import CLASSES, gen_eri, o4, shim  # noqa: F401
from tests.test_grad_tables import X0, qshell_data, run_blob


def contracted(fx, atom, l):
    s = next(s for s in range(fx.nshell) if fx.katom[s] - 1 == atom and
             (fx.Qfinal[s] == 2 if l == 2 else fx.Qstart[s] == 0 and fx.Qfinal[s] == 1 and fx.kprim[s] == 3))
    A, e, c, f0 = qshell_data(fx, s, l)
    if l == 2:
        e, c = np.append(e, 0.45 * e[0]), np.append(c, 0.6 * c[0])
    return s, (A, np.asarray(e), np.asarray(c), f0)


@pytest.mark.parametrize("cls", CLASSES, ids=[gen_eri.tag(c) for c in CLASSES])
def test_folded_gradient_of_contracted_shells(shim, o4, cls):  # noqa: F811
    fx = o4
    rng = np.random.default_rng(11 + sum(cls))
    shells, qs = zip(*(contracted(fx, atom, l) for atom, l in enumerate(cls)))
    Mb = sum(fx.Qfinal[s] for s in shells) + 2
    n = [(l + 1) * (l + 2) // 2 for l in cls]
    dens = [rng.normal(size=(n[i], n[j])) for i, j in ((0, 1), (2, 3), (0, 2), (1, 3), (0, 3), (1, 2))]
    Dab, Dcd, Dac, Dbd, Dad, Dbc = dens
    K = (np.einsum("ab,cd->abcd", Dab, Dcd) - np.einsum("ac,bd->abcd", Dac, Dbd) - np.einsum("ad,bc->abcd", Dad, Dbc))
    ref = run_blob(cls, qs, Mb, K)
    (A, ea, ca, _), (B, eb, cb, _), (C, ec, cc, _), (D, ed, cd, _) = qs
    Fs, geo, ex = [], [], []
    for x, ax in zip(ea, ca):
        for y, by in zip(eb, cb):
            zab, P = x + y, (A * x + B * y) / (x + y)
            Kab = math.exp(-x * y / zab * np.sum((A - B) ** 2)) / zab * ax * by
            for u, cu in zip(ec, cc):
                for v, dv in zip(ed, cd):
                    zcd, Q = u + v, (C * u + D * v) / (u + v)
                    Kcd = math.exp(-u * v / zcd * np.sum((C - D) ** 2)) / zcd * cu * dv
                    inv = 1.0 / (zab + zcd)
                    W = (P * zab + Q * zcd) * inv
                    T = np.sum((P - Q) ** 2) * zab * zcd * inv
                    Fs.append(fmt(Mb, T, exact=True)[:sum(cls) + 2] * X0 * Kab * Kcd * math.sqrt(inv))
                    geo.append(np.concatenate([P - A, W - P, Q - C, W - Q,
                                               [0.5 / zab, 0.5 / zcd, 0.5 * inv, zcd * inv, zab * inv]]))
                    ex.append([x, y, u, v])
    assert len(ex) == math.prod(2 if l == 2 else 3 for l in cls)

    def run(dt, suf, sel):
        a = [np.ascontiguousarray(v, dtype=dt) for v in
             (np.array(Fs)[sel], np.array(geo)[sel], np.array(ex)[sel], np.concatenate([A - B, C - D]), *dens)]
        g = np.zeros(9, dt)
        getattr(shim, f"run{suf}_{gen_eri.tag(cls)}")(len(a[0]), *(v.ctypes.data_as(ctypes.c_void_p) for v in a + [g]))
        return g.astype(np.float64)

    every = slice(None)
    size = sum(np.abs(run(np.float64, "", slice(k, k + 1))).max() for k in range(len(ex)))
    for dt, suf, tol in ((np.float64, "", 1e-11), (np.float32, "_f32", 2e-5)):
        err = np.abs(run(dt, suf, every) - ref).max()
        assert err <= tol * size, (gen_eri.tag(cls), dt, err, size, ref)
