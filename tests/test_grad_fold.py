"""CPU check of the density-folded gradient code (grad_fold.inc).

The generated templates are compiled for the host with g++ and driven, chunk by
chunk as the device kernel does, over the primitive quartets of one shell
quartet on four distinct oxygen centres; the nine derivative sums are compared
with the table-driven gradient program of the same class.  Both evaluate the
same integrals in FP64 with sums of a few thousand terms, so they agree to
1e-11 of the largest derivative; the FP32 form carries the rounding of single
precision (6e-8) over the same sums and is held to 2e-5.
"""
import ctypes
import math
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "quick_amd" / "csrc"
sys.path.insert(0, str(CSRC))
import gen_eri  # noqa: E402
import gen_gradw  # noqa: E402
from tests.test_grad_tables import X0, qshell_data, run_blob  # noqa: E402

from oracle.oracle import fmt  # noqa: E402

CLASSES = list(gen_gradw.FOLD_CLASSES)


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("gf")
    gen_gradw.write(str(d / "grad_fold.inc"))
    src = ["#define __device__", "#define __forceinline__ inline", '#include "grad_fold.inc"', """
template <class Fd, int K, class R>
static void chunk(int np, int nf, const R* F, const R* geo, const R* ex, const R* ABCD, const R* const* D, R* g) {
    R W[Fd::kW[K]] = {}, S[Fd::kS[K] + 1] = {}, tab[3] = {}, tcd[3] = {};
    const R *AB = ABCD, *CD = ABCD + 3;
    Fd::template fold<K, R>(D[0], D[1], D[2], D[3], D[4], D[5], AB[0], AB[1], AB[2], CD[0], CD[1], CD[2], W);
    for (int p = 0; p < np; ++p) {
        const R* G = geo + 17 * p;
        R u[10] = {};
        Fd::template vrr<K, R>(F + nf * p, G[0], G[1], G[2], G[3], G[4], G[5], G[6], G[7], G[8], G[9], G[10], G[11],
                               G[12], G[13], G[14], G[15], G[16], W, S, u);
        const R al = ex[4 * p], be = ex[4 * p + 1], ga = ex[4 * p + 2], de = ex[4 * p + 3], eta = ga + de;
        for (int x = 0; x < 3; ++x) {
            g[x] += 2 * al * u[x] - u[4 + x];
            g[3 + x] += 2 * be * (u[x] + AB[x] * u[3]);
            g[6 + x] += ga / eta * (u[4 + x] + u[7 + x] - 2 * (al + be) * u[x] - 2 * (be * AB[x] + de * CD[x]) * u[3]) -
                        u[7 + x];
        }
    }
    Fd::template end<K, R>(D[0], D[1], D[2], D[3], D[4], D[5], AB[0], AB[1], AB[2], CD[0], CD[1], CD[2], S, tab, tcd);
    for (int x = 0; x < 3; ++x) { g[x] += tab[x]; g[3 + x] -= tab[x]; g[6 + x] += tcd[x]; }
}"""]
    for cls in CLASSES:
        t = gen_eri.tag(cls)
        for R, suf, fd in (("double", "", f"Fold_{t}"), ("float", "_f32", f"Fold_{t}_f")):
            calls = "\n".join(f"    if constexpr ({fd}::kChunks > {k}) chunk<{fd}, {k} < {fd}::kChunks ? {k} : 0, {R}>"
                              "(np, nf, F, geo, ex, ABCD, D, g);" for k in range(16))
            src.append(f"""extern "C" void run{suf}_{t}(int np, const {R}* F, const {R}* geo, const {R}* ex,
                        const {R}* ABCD, const {R}* D0, const {R}* D1, const {R}* D2, const {R}* D3, const {R}* D4,
                        const {R}* D5, {R}* g) {{
    const {R}* D[6] = {{D0, D1, D2, D3, D4, D5}};
    const int nf = {sum(cls) + 2};
    for (int k = 0; k < 9; ++k) g[k] = 0;
{calls}
}}""")
    (d / "shim.cpp").write_text("\n".join(src) + "\n")
    so = d / "shim.so"
    subprocess.run(["g++", "-O0", "-fPIC", "-shared", "-std=c++17", "-I", str(d), str(d / "shim.cpp"), "-o", str(so)],
                   check=True)
    return ctypes.CDLL(str(so))


@pytest.fixture(scope="module")
def o4():
    from quick_amd.basis import build_basis
    xyz = np.array([[0.0, 0.0, 0.0], [1.3, 0.1, 0.0], [0.5, 1.2, 0.2], [0.6, 0.5, 1.1]])
    return build_basis(["O"] * 4, xyz)


@pytest.mark.parametrize("cls", CLASSES, ids=[gen_eri.tag(c) for c in CLASSES])
def test_folded_gradient_code_matches_table_program(shim, o4, cls):
    fx = o4
    rng = np.random.default_rng(7 + sum(cls))
    shells = []
    for atom, l in enumerate(cls):
        cand = [s for s in range(fx.nshell) if fx.katom[s] - 1 == atom and fx.Qstart[s] <= l <= fx.Qfinal[s]]
        shells.append(cand[len(cand) // 2])   # a contracted shell: several primitive quartets
    qs = [qshell_data(fx, s, L) for s, L in zip(shells, cls)]
    Mb = sum(fx.Qfinal[s] for s in shells) + 2
    n = [(l + 1) * (l + 2) // 2 for l in cls]
    Dab, Dcd, Dac, Dbd, Dad, Dbc = (rng.normal(size=(n[i], n[j])) for i, j in
                                    ((0, 1), (2, 3), (0, 2), (1, 3), (0, 3), (1, 2)))
    K = (np.einsum("ab,cd->abcd", Dab, Dcd) - np.einsum("ac,bd->abcd", Dac, Dbd) - np.einsum("ad,bc->abcd", Dad, Dbc))
    ref = run_blob(cls, qs, Mb, K)
    (A, ea, ca, _), (B, eb, cb, _), (C, ec, cc, _), (D, ed, cd, _) = qs
    Fs, geo, ex = [], [], []
    for x, ax in zip(ea, ca):
        for y, by in zip(eb, cb):
            zab = x + y
            P = (A * x + B * y) / zab
            Kab = math.exp(-x * y / zab * np.sum((A - B) ** 2)) / zab * ax * by
            for u, cu in zip(ec, cc):
                for v, dv in zip(ed, cd):
                    zcd = u + v
                    Q = (C * u + D * v) / zcd
                    Kcd = math.exp(-u * v / zcd * np.sum((C - D) ** 2)) / zcd * cu * dv
                    inv = 1.0 / (zab + zcd)
                    W = (P * zab + Q * zcd) * inv
                    T = np.sum((P - Q) ** 2) * zab * zcd * inv
                    Fs.append(fmt(Mb, T, exact=True)[:sum(cls) + 2] * X0 * Kab * Kcd * math.sqrt(inv))
                    geo.append(np.concatenate([P - A, W - P, Q - C, W - Q,
                                               [0.5 / zab, 0.5 / zcd, 0.5 * inv, zcd * inv, zab * inv]]))
                    ex.append([x, y, u, v])
    args = [np.array(Fs), np.array(geo), np.array(ex), np.concatenate([A - B, C - D]), Dab, Dcd, Dac, Dbd, Dad, Dbc]
    scale = np.abs(ref).max()
    assert scale > 1e-10
    for dt, suf, tol in ((np.float64, "", 1e-11 * max(1.0, scale)), (np.float32, "_f32", 2e-5 * scale)):
        a = [np.ascontiguousarray(v, dtype=dt) for v in args]
        g = np.zeros(9, dt)
        p = [v.ctypes.data_as(ctypes.c_void_p) for v in a + [g]]
        getattr(shim, f"run{suf}_{gen_eri.tag(cls)}")(len(Fs), *p)
        err = np.abs(g.astype(np.float64) - ref).max()
        assert err <= tol, (gen_eri.tag(cls), dt, err, scale, g, ref)
