"""A CPU build of the library's Fock, gradient, one-electron and work-list code.

The device sources are compiled with g++ against the headers in include/ (see
emulator.cpp): the same kernels and the same host code, with every device
allocation and a block's dynamic LDS lying against inaccessible pages.  Text
that only the device compiler takes (inline asm that hides a value from the
optimiser, the declaration of dynamic LDS, the launch by address) is replaced in
copies, and the work lists, which share one allocation on the device, get one each.  Classes with a d shell are left out of the two-electron part, to keep
the build short: their launchers stop the process.
"""
from __future__ import annotations

import copy
import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import numpy as np

HERE = Path(__file__).resolve().parent
ROOT = HERE.parents[1]
CSRC = ROOT / "quick_amd" / "csrc"


def _host_text(text: str) -> str:
    text = re.sub(r"asm volatile\([^;]*\);", ";", text)
    text = re.sub(r"extern __shared__ (?:__align__\(\d+\) )?([\w ]+?) (\w+)\[\];",
                  r"\1* const \2 = (\1*)emu::dynamic_lds();", text)
    text = text.replace("(void)hipLaunchKernel(f, dim3(grid), dim3(256), args, lds, s);",
                        "emu_launch_kernel((void (*)(FockArgs, ClassWork))f, dim3(grid), dim3(256), lds, s, aa, ww);")
    # each work list in an allocation of its own instead of one for all
    text = text.replace("b.view(reinterpret_cast<T*>(mem.p + off[slot]), count);", "b.release(); (void)b.alloc(count);")
    return text


def build(out: Path, jobs: int = 8) -> Path:
    """compiles into the directory `out`; returns the shared library"""
    src, gen = out / "quick_amd" / "csrc", out / "quick_amd" / "csrc" / "gen"
    gen.mkdir(parents=True)
    (out / "include").mkdir()
    (out / "include" / "quick_mi355x.h").write_text((ROOT / "include" / "quick_mi355x.h").read_text())
    for f in list(CSRC.glob("*.hip")) + list(CSRC.glob("*.h")) + list(CSRC.glob("*.cpp")):
        (src / f.name).write_text(_host_text(f.read_text()))
    for code, args in (
            ("import gen_eri as g, sys; g.main(sys.argv[1]); g.write_units(sys.argv[2]); g.write_team(sys.argv[3])",
             ("eri_generated.inc", "gen", "team_tables.inc")),
            ("import gen_grad as g, sys; g.write(sys.argv[1])", ("grad_tables.inc",)),
            ("import gen_gradw as g, sys; g.write(sys.argv[1]); g.write_units(sys.argv[2])", ("grad_fold.inc", "gen"))):
        subprocess.run([sys.executable, "-c", code, *(str(src / a) for a in args)], check=True,
                       env={**os.environ, "PYTHONPATH": str(CSRC)}, stdout=subprocess.DEVNULL)
    units = [src / n for n in ("qk_fock.hip", "qk_lists.hip", "qk_oneint.hip", "qk_grad.hip", "qk_host.cpp")]
    units += [HERE / "emulator.cpp"] + list(gen.glob("*.hip"))
    units.sort(key=lambda u: -u.stat().st_size)   # the longest compilations first

    def compile_(u: Path) -> Path:
        obj = out / (u.stem + ".o")
        subprocess.run(["g++", "-x", "c++", "-std=c++17", "-O1", "-fPIC", "-w", "-I",
                        str(HERE / "include"), "-I", str(src), "-c", str(u), "-o", str(obj)], check=True)
        return obj

    with ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(compile_, units))
    # whatever is left undefined in the library's own name space stops the process
    table = subprocess.run(["nm", *map(str, objs)], check=True, capture_output=True, text=True).stdout
    have = {p[-1] for p in map(str.split, table.splitlines()) if len(p) == 3}
    want = {p[-1] for p in map(str.split, table.splitlines()) if len(p) == 2 and p[0] == "U"} - have
    want |= {"qk_scf", "qk_scf_default_opts"} - have   # bound by quick_amd.fock
    stubs = sorted(s for s in want if s.startswith(("_ZN2qk", "qk_", "_Z17qk_", "launch_")))
    (out / "stubs.s").write_text("".join(f".globl {s}\n{s}:\n" for s in stubs) + " ud2\n" +
                                 '.section .note.GNU-stack,"",@progbits\n')
    lib = out / "libquick_emulated.so"
    subprocess.run(["g++", "-shared", "-o", str(lib), *map(str, objs), str(out / "stubs.s"), "-ldl"], check=True)
    return lib


def symbols(lib: Path) -> list[str]:
    """the functions the library exports"""
    txt = subprocess.run(["nm", "-D", "--defined-only", str(lib)], check=True, capture_output=True, text=True).stdout
    return [line.split()[-1] for line in txt.splitlines() if line.split()[-2] in "TWtwVu"]


def run(lib: Path, code: str, low: bool = False, timeout: int = 600) -> str:
    """runs `code` in a child process whose quick_amd loads the emulated library"""
    env = {**os.environ, "QUICK_MI355X_LIB": str(lib), "OMP_NUM_THREADS": "1"}
    pre = ("import faulthandler, sys; faulthandler.enable(); sys.modules['torch'] = None\n"
           "import ctypes as C, numpy as np\nfrom quick_amd.fock import *\nfrom quick_amd.fock import _ptr\n"
           f"emu = C.CDLL({str(lib)!r}); emu.emu_record.restype = C.c_char_p; emu.emu_alloc_low({int(low)})\n")
    p = subprocess.run([sys.executable, "-"], input=pre + code, cwd=ROOT, env=env, capture_output=True, text=True,
                       timeout=timeout)
    assert p.returncode == 0, f"exit {p.returncode}\n{p.stdout[-2000:]}\n{p.stderr[-4000:]}"
    return p.stdout


def without_d(b):
    """a copy of the basis without its d shells"""
    keep = [s for s in range(b.nshell) if b.Qfinal[s] < 2]
    fns = [f for s in keep for f in range(b.ksumtype[s] - 1, b.ksumtype[s + 1] - 1)]
    c = copy.copy(b)
    n = [b.ksumtype[s + 1] - b.ksumtype[s] for s in keep]
    c.nshell, c.nbasis = len(keep), len(fns)
    for k in ("kstart", "kprim", "katom", "ktype", "Qstart", "Qfinal"):
        setattr(c, k, np.asarray(getattr(b, k))[keep])
    for k in ("Qsbasis", "Qfbasis"):
        setattr(c, k, np.asarray(getattr(b, k))[keep])
    c.ksumtype = np.concatenate([[1], 1 + np.cumsum(n)]).astype(np.int32)
    c.KLMN, c.cons = b.KLMN[:, fns], b.cons[fns]
    c.gccoeff, c.gcexpo = b.gccoeff[:, fns], b.gcexpo[:, fns]
    return c
