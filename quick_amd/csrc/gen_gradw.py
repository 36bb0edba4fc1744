"""Generator of the density-folded gradient code (grad_fold.inc).

One contracted quartet (ab|cd) contributes sum K_abcd d(ab|cd)/dR to the
gradient, with the density factors

    K = w (4 D_ab D_cd - h (D_ac D_bd + D_ad D_bc)).

The horizontal recurrence is linear with coefficients that depend on the
geometry alone, so its adjoint is applied to K once per contracted quartet:

    W_ef = sum_abcd B(ab -> e; A-B) C(cd -> f; C-D) K_abcd,
    sum K (ab|cd) = sum W_ef [e0|f0].

With the functions on A and C only, the derivatives of a primitive [e0|f0] are

    d/dA_x = 2 alpha [e+1x|f] - e_x [e-1x|f],
    d/dB_x = 2 beta ([e+1x|f] + (A-B)_x [e|f]),
    d/dC_x = 2 gamma [e|f+1x] - f_x [e|f-1x],

and translational invariance (the electron-transfer relation) replaces the one
quantity raised on the ket:

    2 eta [e|f+1x] = e_x [e-1x|f] + f_x [e|f-1x] - 2 zeta [e+1x|f]
                     - 2 (beta (A-B)_x + delta (C-D)_x) [e|f].

So a primitive quartet needs ten sums over (e, f) with the weights W,

    U_x = sum W [e+1x|f],  E = sum W [e|f],
    L_x = sum W e_x [e-1x|f],  M_x = sum W f_x [e|f-1x],

of a recurrence raised by one on the bra alone, instead of four contracted sets
raised on both sides with a derivative recurrence and a contraction each.  W
itself depends on A-B and C-D: those terms need the contracted [e0|f0] below
the top of the recurrence only (S), and none for an s function on B and D.

Per class and chunk of the ket functions f (a chunk bounds the weights and
sums a lane holds) this emits, as templates over the arithmetic type:

    gf_fold:  density blocks -> W of the chunk
    gf_vrr:   recurrence of one primitive quartet: the ten sums, and S += [e|f]
    gf_end:   the terms of dW/d(A-B) and dW/d(C-D), from S and the density blocks
"""
from __future__ import annotations

import itertools
import math
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from gen_eri import QUICK_ORDER, erange, first_dir, name_of, sub, tag  # noqa: E402

X = "xyz"

# Classes evaluated this way: per precision (FP64, FP32) the largest number of
# ket functions f per chunk and the wavefronts per SIMD the kernel is built for.
# More functions per chunk share more of the recurrence; the weights, sums and
# intermediates of a chunk have to fit the registers (256 FP64 values at one
# wavefront per SIMD), or the primitive loop runs on scratch memory.  Measured
# per class on n-icosane (FP64) and (H2O)32 (FP32 below 1e-3), kernel times in
# ms at (chunk, waves): pppp FP64 (9, 1) 1.46, (4, 1) 0.83, (4, 2) 2.28; ddpp
# FP64 (4, 1) 1.83, (2, 1) 1.17, (1, 1) 0.64; dddp FP64 (2, 1) 1.54, (1, 1)
# 0.98; dppp FP64 (9, 1) 5.2, (4, 1) 2.87, (3, 1) 2.42, (2, 2) 4.84; dsps FP64
# (3, 1) 1.90, (3, 2) 1.34; dspp FP32 (9, 1) 0.84, (9, 2) 0.56.
FOLD_CLASSES = {
    (0, 0, 0, 0): ((1, 1), (1, 1)), (1, 0, 0, 0): ((1, 1), (1, 1)), (1, 0, 1, 0): ((3, 1), (3, 1)),
    (1, 1, 0, 0): ((1, 1), (1, 1)), (1, 1, 1, 0): ((3, 1), (3, 3)), (1, 1, 1, 1): ((4, 1), (4, 2)),
    (2, 0, 0, 0): ((1, 1), (1, 1)), (2, 0, 1, 0): ((3, 2), (3, 2)), (2, 0, 1, 1): ((6, 1), (9, 2)),
    (2, 0, 2, 0): ((6, 1), (6, 2)), (2, 1, 0, 0): ((1, 2), (1, 2)), (2, 1, 1, 0): ((3, 1), (3, 2)),
    (2, 1, 1, 1): ((3, 1), (3, 2)), (2, 1, 2, 0): ((3, 1), (3, 2)), (2, 1, 2, 1): ((2, 1), (4, 1)),
    (2, 2, 0, 0): ((1, 1), (1, 3)), (2, 2, 1, 0): ((2, 1), (2, 2)), (2, 2, 1, 1): ((1, 1), (3, 1)),
    (2, 2, 2, 0): ((1, 1), (3, 1)), (2, 2, 2, 1): ((1, 1), (2, 1)),
}


def up(v, x, n=1):
    w = list(v)
    w[x] += n
    return tuple(w)


def transfer(l1, l2):
    """(ab) -> e coefficients: for each (a, b) of the shell pair a list of
    (e, power triple of the centre difference, integer)"""
    out = {}
    for a in QUICK_ORDER[l1]:
        for b in QUICK_ORDER[l2]:
            t = []
            for k in itertools.product(*(range(v + 1) for v in b)):
                c = math.prod(math.comb(b[i], k[i]) for i in range(3))
                t.append((tuple(a[i] + k[i] for i in range(3)), tuple(b[i] - k[i] for i in range(3)), c))
            out[a, b] = t
    return out


def chunks(cls, most):
    """the ket functions in groups of at most `most`, those lowered to the same
    function together"""
    F = erange(cls[2], cls[2] + cls[3])
    fam = {}
    for f in F:
        key = f if sum(f) == cls[2] else sub(f, first_dir(f))
        fam.setdefault(key, []).append(f)
    out = []
    for g in fam.values():
        for i in range(0, len(g), most):
            part = g[i:i + most]
            if out and len(out[-1]) + len(part) <= most:
                out[-1] += part
            else:
                out.append(part)
    return out


def s_needed(cls, part):
    """(e, f) of the chunk whose contracted value dW/d(A-B) or dW/d(C-D) needs"""
    la, lb, lc, ld = cls
    need = []
    for f in part:
        for e in erange(la, la + lb):
            if (lb and sum(e) < la + lb) or (ld and sum(f) < lc + ld):
                need.append((e, f))
    return need


def power(base, p):
    """product of powers of the components base0..2 as an expression, '' for 1"""
    return " * ".join(f"{base}{X[i]}" for i in range(3) for _ in range(p[i]))


def term(coef, *factors):
    f = [x for x in factors if x]
    if coef != 1:
        f = [f"R({coef})"] + f
    return " * ".join(f) if f else "R(1)"


def blocks(cls):
    nA, nB, nC, nD = (len(QUICK_ORDER[l]) for l in cls)
    return nA, nB, nC, nD


def gen_rows(cls, part, body):
    """lines that form, for each (a, b), the density factors k<cd> and the ket
    transfer t<f> = sum_cd C(cd -> f) K of the chunk, then body(a, b, ia, ib)"""
    la, lb, lc, ld = cls
    nA, nB, nC, nD = blocks(cls)
    ket = transfer(lc, ld)
    lines = []
    for ia, a in enumerate(QUICK_ORDER[la]):
        for ib, b in enumerate(QUICK_ORDER[lb]):
            lines.append("    {")
            used = {}
            for ic, c in enumerate(QUICK_ORDER[lc]):
                for id_, d in enumerate(QUICK_ORDER[ld]):
                    if any(e in part for e, _, _ in ket[c, d]):
                        used[c, d] = f"k{ic}_{id_}"
                        lines.append(f"        const R k{ic}_{id_} = Dab[{ia * nB + ib}] * Dcd[{ic * nD + id_}] - "
                                     f"(Dac[{ia * nC + ic}] * Dbd[{ib * nD + id_}] + Dad[{ia * nD + id_}] * Dbc[{ib * nC + ic}]);")
            for kf, f in enumerate(part):
                t = [term(n, power("CD", p), used[cd]) for cd, lst in ket.items() for e, p, n in lst if e == f]
                lines.append(f"        const R t{kf} = {' + '.join(t)};")
            lines += ["        " + s for s in body(a, b, used)]
            lines.append("    }")
    return lines


ARGS_D = "const R* Dab, const R* Dcd, const R* Dac, const R* Dbd, const R* Dad, const R* Dbc"
ARGS_G = "R ABx, R ABy, R ABz, R CDx, R CDy, R CDz"


def gen_fold(cls, k, part):
    la, lb, _, _ = cls
    E = erange(la, la + lb)
    eix = {e: i for i, e in enumerate(E)}
    bra = transfer(la, lb)
    nf = len(part)

    def body(a, b, used):
        return [f"W[{eix[e] * nf + kf}] += {term(n, power('AB', p), f't{kf}')};" for kf in range(nf)
                for e, p, n in bra[a, b]]

    head = (f"template <typename R>\n__device__ __forceinline__ void gf_fold_{tag(cls)}_{k}({ARGS_D}, {ARGS_G}, R* W)")
    return f"{head}\n{{\n" + "\n".join(gen_rows(cls, part, body)) + "\n}\n"


def vrr_order(cls, part):
    """the recurrence's nodes in dependency order, and the targets"""
    la, lb, lc, ld = cls
    E = erange(la, la + lb)
    targets = []
    for f in part:
        for e in erange(max(la - 1, 0), la + lb + 1):
            targets.append((e, f, 0))
        for x in range(3):
            if f[x]:
                targets += [(e, sub(f, x), 0) for e in E]
    order, seen = [], set()

    def visit(node):
        if node in seen:
            return
        e, f, m = node
        deps = []
        if sum(f) > 0:
            i = first_dir(f)
            f1 = sub(f, i)
            deps += [(e, f1, m), (e, f1, m + 1)]
            if f1[i] > 0:
                deps += [(e, sub(f1, i), m), (e, sub(f1, i), m + 1)]
            if e[i] > 0:
                deps.append((sub(e, i), f1, m + 1))
        elif sum(e) > 0:
            i = first_dir(e)
            e1 = sub(e, i)
            deps += [(e1, f, m), (e1, f, m + 1)]
            if e1[i] > 0:
                deps += [(sub(e1, i), f, m), (sub(e1, i), f, m + 1)]
        for d in deps:
            visit(d)
        seen.add(node)
        order.append(node)

    for t in targets:
        visit(t)
    return order


def gen_vrr(cls, k, part):
    la, lb, lc, ld = cls
    E = erange(la, la + lb)
    eix = {e: i for i, e in enumerate(E)}
    fix = {f: i for i, f in enumerate(part)}
    nf = len(part)
    six = {s: i for i, s in enumerate(s_needed(cls, part))}
    w = lambda e, f: f"W[{eix[e] * nf + fix[f]}]"
    lines, flops = [], 0
    for node in vrr_order(cls, part):
        e, f, m = node
        nm = name_of(e, f, m)
        if sum(e) == 0 and sum(f) == 0:
            lines.append(f"    const R {nm} = F[{m}];")
        else:
            if sum(f) > 0:
                i = first_dir(f)
                f1 = sub(f, i)
                expr = f"QC{X[i]} * {name_of(e, f1, m)} + WQ{X[i]} * {name_of(e, f1, m + 1)}"
                flops += 3
                if f1[i] > 0:
                    f2 = sub(f1, i)
                    expr += f" + R({f1[i]}) * oo2e * ({name_of(e, f2, m)} - roe * {name_of(e, f2, m + 1)})"
                    flops += 5
                if e[i] > 0:
                    expr += f" + R({e[i]}) * oo2ze * {name_of(sub(e, i), f1, m + 1)}"
                    flops += 3
            else:
                i = first_dir(e)
                e1 = sub(e, i)
                expr = f"PA{X[i]} * {name_of(e1, f, m)} + WP{X[i]} * {name_of(e1, f, m + 1)}"
                flops += 3
                if e1[i] > 0:
                    e2 = sub(e1, i)
                    expr += f" + R({e1[i]}) * oo2z * ({name_of(e2, f, m)} - roz * {name_of(e2, f, m + 1)})"
                    flops += 5
            lines.append(f"    const R {nm} = {expr};")
        if m:
            continue
        # the sums this value enters, taken as soon as it exists
        if f in fix:
            for x in range(3):
                if e[x] and sub(e, x) in eix:
                    lines.append(f"    u[{x}] += {w(sub(e, x), f)} * {nm};")
                    flops += 2
            if e in eix:
                lines.append(f"    u[3] += {w(e, f)} * {nm};")
                flops += 2
            for x in range(3):
                if up(e, x) in eix:
                    lines.append(f"    u[{4 + x}] += {term(e[x] + 1, w(up(e, x), f))} * {nm};")
                    flops += 2 + (e[x] > 0)
            if (e, f) in six:
                lines.append(f"    S[{six[e, f]}] += {nm};")
                flops += 1
        if e in eix:
            for x in range(3):
                if up(f, x) in fix:
                    lines.append(f"    u[{7 + x}] += {term(f[x] + 1, w(e, up(f, x)))} * {nm};")
                    flops += 2 + (f[x] > 0)
    head = (f"template <typename R>\n__device__ __forceinline__ void gf_vrr_{tag(cls)}_{k}(const R* F, R PAx, R PAy, R PAz, "
            "R WPx, R WPy, R WPz, R QCx, R QCy, R QCz, R WQx, R WQy, R WQz, R oo2z, R oo2e, R oo2ze, R roz, R roe, "
            "const R* W, R* S, R* u)")
    return f"{head}\n{{\n" + "\n".join(lines) + "\n}\n", flops


def gen_end(cls, k, part):
    """tab[x] += sum K d(ab -> e)/d(A-B)_x S, tcd[x] += the same in C-D"""
    la, lb, lc, ld = cls
    six = {s: i for i, s in enumerate(s_needed(cls, part))}
    bra, ket = transfer(la, lb), transfer(lc, ld)

    def body(a, b, used):
        out = []
        for x in range(3):
            if b[x]:   # d(a b|/d(A-B)_x = b_x (a b-1x|
                low = sub(b, x)
                for kf, f in enumerate(part):
                    v = [term(n, power("AB", p), f"S[{six[e, f]}]") for e, p, n in transfer_one(a, low)]
                    out.append(f"tab[{x}] += {term(b[x], f't{kf}')} * ({' + '.join(v)});")
        if ld:
            low_f = [f for f in part if sum(f) < lc + ld]
            for f in low_f:
                v = [term(n, power("AB", p), f"S[{six[e, f]}]") for e, p, n in bra[a, b]]
                nm = f"h{part.index(f)}"
                out.append(f"const R {nm} = {' + '.join(v)};")
            for (c, d), kn in used.items():
                for f, p, n in ket[c, d]:
                    if f not in low_f:
                        continue
                    for x in range(3):
                        if p[x]:
                            out.append(f"tcd[{x}] += {term(n * p[x], power('CD', sub(p, x)), kn)} * h{part.index(f)};")
        return out

    rows = gen_rows(cls, part, body) if six else []
    head = (f"template <typename R>\n__device__ __forceinline__ void gf_end_{tag(cls)}_{k}({ARGS_D}, {ARGS_G}, "
            "const R* S, R* tab, R* tcd)")
    return f"{head}\n{{\n" + "\n".join(rows) + "\n}\n"


def transfer_one(a, b):
    return [(tuple(a[i] + k[i] for i in range(3)), tuple(b[i] - k[i] for i in range(3)),
             math.prod(math.comb(b[i], k[i]) for i in range(3)))
            for k in itertools.product(*(range(v + 1) for v in b))]


def class_code(cls, most, suffix):
    """code and chunk traits of one class and precision; suffix names the chunking"""
    parts = chunks(cls, most)
    nE = len(erange(cls[0], cls[0] + cls[1]))
    out, flops = [], 0
    for k, part in enumerate(parts):
        name = f"{suffix}{k}"
        v, fl = gen_vrr(cls, name, part)
        out += [gen_fold(cls, name, part), v, gen_end(cls, name, part)]
        flops += fl
    return out, parts, [nE * len(p) for p in parts], [len(s_needed(cls, p)) for p in parts], flops


def write(path):
    out = ["// Generated by quick_amd/csrc/gen_gradw.py -- do not edit.",
           "// Density-folded gradient code per class and chunk of ket functions (gf_fold, gf_vrr, gf_end).",
           "#pragma once", ""]
    for cls, (f64, f32) in FOLD_CLASSES.items():
        t = tag(cls)
        forms = {"": f64} if f64 == f32 else {"": f64, "f": f32}
        for suf, (most, waves) in forms.items():
            code, parts, nw, ns, _ = class_code(cls, most, suf)
            out += code
            out.append(f"struct Fold_{t}{'_' + suf if suf else ''} {{")
            out.append(f"    static constexpr int kChunks = {len(parts)}, kWaves = {waves};")
            out.append(f"    static constexpr int kW[{len(parts)}] = {{{', '.join(map(str, nw))}}};")
            out.append(f"    static constexpr int kS[{len(parts)}] = {{{', '.join(map(str, ns))}}};")
            for fn, args, call in (
                    ("fold", f"{ARGS_D}, {ARGS_G}, R* W", "Dab, Dcd, Dac, Dbd, Dad, Dbc, ABx, ABy, ABz, CDx, CDy, CDz, W"),
                    ("vrr", "const R* F, R PAx, R PAy, R PAz, R WPx, R WPy, R WPz, R QCx, R QCy, R QCz, R WQx, R WQy, "
                     "R WQz, R oo2z, R oo2e, R oo2ze, R roz, R roe, const R* W, R* S, R* u",
                     "F, PAx, PAy, PAz, WPx, WPy, WPz, QCx, QCy, QCz, WQx, WQy, WQz, oo2z, oo2e, oo2ze, roz, roe, W, S, u"),
                    ("end", f"{ARGS_D}, {ARGS_G}, const R* S, R* tab, R* tcd",
                     "Dab, Dcd, Dac, Dbd, Dad, Dbc, ABx, ABy, ABz, CDx, CDy, CDz, S, tab, tcd")):
                out.append("    template <int K, typename R>")
                out.append(f"    static __device__ __forceinline__ void {fn}({args}) {{")
                for k in range(len(parts)):
                    out.append(f"        {'if' if k == 0 else 'else if'} constexpr (K == {k}) gf_{fn}_{t}_{suf}{k}<R>({call});")
                out.append("    }")
            out.append("};")
        if len(forms) == 1:
            out.append(f"using Fold_{t}_f = Fold_{t};")
    new = "\n".join(out) + "\n"
    if not os.path.exists(path) or open(path).read() != new:
        open(path, "w").write(new)


def write_units(outdir):
    """one translation unit per class"""
    os.makedirs(outdir, exist_ok=True)
    for cls in FOLD_CLASSES:
        t, args = tag(cls), ", ".join(map(str, cls))
        body = ["// Generated by quick_amd/csrc/gen_gradw.py -- do not edit.", '#include "../qk_grad_light.h"',
                "namespace qk {"]
        for suf, R in (("", "double"), ("f32_", "float")):
            body += [f"void launch_grad_light_{suf}{t}(const GradArgs& a, const ClassWork& w, int grid, size_t lds, "
                     "hipStream_t s) {",
                     "    static const long long cap = scratch_grid_cap(kernel_scratch(reinterpret_cast<const void*>("
                     f"&grad_light_kernel<{args}, {R}>)), 4);",
                     f"    hipLaunchKernelGGL((grad_light_kernel<{args}, {R}>), dim3((int)std::min<long long>(grid, cap)), "
                     "dim3(256), lds, s, a, w);", "}"]
        body.append("}  // namespace qk")
        fn = os.path.join(outdir, f"grad_{t}.hip")
        new = "\n".join(body) + "\n"
        if not os.path.exists(fn) or open(fn).read() != new:
            open(fn, "w").write(new)


if __name__ == "__main__":
    if len(sys.argv) > 1:
        write(sys.argv[1])
        write_units(os.path.join(os.path.dirname(sys.argv[1]), "gen"))
    else:
        for cls, forms in FOLD_CLASSES.items():
            for most in sorted({m for m, _ in forms}):
                code, parts, nw, ns, fl = class_code(cls, most, "")
                print(tag(cls), "chunk", most, "passes", len(parts), "W", nw, "S", ns, "nodes",
                      [len(vrr_order(cls, p)) for p in parts], "flops", fl)
