"""The order of the XC GEMM tasks over the XCDs (csrc/qk_xc_deal.h), compiled for
the host: every task goes out exactly once, and no XCD is left with much more
than its share, whether a chunk has one batch or hundreds."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
SRC = r"""
#include "qk_xc_deal.h"
#include <cstdio>
struct T4 { int b, i, j, pad; };
int main() {   // per chunk: number of batches, then the column tiles of each
    qk::XcDeal<T4> deal;
    int nb;
    while (std::scanf("%d", &nb) == 1) {
        std::vector<T4> out[2];
        for (int b = 0; b < nb; ++b) {
            int T;
            if (std::scanf("%d", &T) != 1) return 1;
            deal.begin_batch();
            for (int r = 0; r < 4; ++r)
                for (int c = 0; c < T; ++c) deal.rho(T4{b, r, c, 0});
            for (int I = 0; I < T; ++I)
                for (int J = 0; J <= I; ++J) deal.v(T4{b, I, J, 0});
        }
        deal.finish(out[0], out[1]);
        for (auto& o : out) {
            for (const T4& t : o) std::printf("%d %d %d ", t.b, t.i, t.j);
            std::printf("\n");
        }
    }
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("deal")
    (d / "deal.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(ROOT / "quick_amd" / "csrc"), str(d / "deal.cpp"), "-o",
                    str(d / "deal")], check=True)

    def run(chunks):
        text = "\n".join(f"{len(c)} " + " ".join(map(str, c)) for c in chunks)
        out = subprocess.run([str(d / "deal")], input=text, capture_output=True, text=True, check=True).stdout
        rows = [np.array(r.split(), int).reshape(-1, 3) for r in out.split("\n")[:-1]]
        return list(zip(rows[::2], rows[1::2]))

    return run


CHUNKS = {"1x25": [25], "1x1": [1], "2x11": [11, 11], "8x4": [4] * 8, "8-mixed": [25, 25, 22, 18, 14, 12, 10, 9],
          "16x3": [3] * 16, "125-mixed": [25 - b % 20 for b in range(125)], "512x5": [5] * 512,
          "600-mixed": [1 + b % 9 for b in range(600)]}


def test_every_task_once_and_no_xcd_overloaded(deal):
    chunks = list(CHUNKS.values())
    for (name, T), (rho, v) in zip(CHUNKS.items(), deal(chunks)):
        want = [{(b, r, c) for b, t in enumerate(T) for r in range(4) for c in range(t)},
                {(b, i, j) for b, t in enumerate(T) for i in range(t) for j in range(i + 1)}]
        for kind, got, tasks in zip(("rho", "v"), (rho, v), want):
            real = [tuple(t) for t in got.tolist() if t[0] >= 0]
            assert len(real) == len(tasks) and set(real) == tasks, (name, kind)
            load = [sum(1 for t in got[x::8].tolist() if t[0] >= 0) for x in range(8)]
            # at most a task a CU, or within a quarter of an even share
            assert max(load) <= max(32, 1 + 1.25 * len(tasks) / 8), (name, kind, load)
