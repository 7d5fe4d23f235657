"""The rule by which mt_gemm_noalloc_f32 takes or refuses a call stands by itself
(csrc/noalloc_rule.hpp): nothing of the planner goes into it, and its answers on
both sides of recorded limits stay what they were."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

RULE = Path(__file__).resolve().parent.parent / "minitensor_amd" / "csrc" / "noalloc_rule.hpp"
# M, N, K, batch, compute units: taken at K or not; the other way at K - 1
EDGES = [(732, 1694, 6241, 1, 256, 0), (377, 8540, 1761, 1, 256, 1), (1785, 10131, 1249, 3, 256, 1),
         (5923, 440, 1361, 1, 256, 0), (220, 9031, 577, 3, 304, 1), (4360, 333, 2881, 1, 304, 0),
         (732, 5682, 3425, 1, 304, 0), (1834, 510, 1361, 3, 256, 0)]
MAIN = """#include <cstdio>
#include "noalloc_rule.hpp"
int main() {
    long m, n, k, b;
    int cus;
    while (std::scanf("%ld %ld %ld %ld %d", &m, &n, &k, &b, &cus) == 5)
        std::printf("%d\\n", (int)noalloc_rule::takes(m, n, k, b, cus, (size_t)32 << 20));
}
"""


def test_rule_uses_nothing_of_the_planner():
    assert re.findall(r'#include\s+"', RULE.read_text()) == []


def test_recorded_answers(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    (tmp_path / "rule.cpp").write_text(MAIN)
    subprocess.run([cxx, "-O1", "-std=c++17", f"-I{RULE.parent}", str(tmp_path / "rule.cpp"), "-o",
                    str(tmp_path / "rule")], check=True)
    sizes = [(m, n, k - d, b, c) for m, n, k, b, c, _ in EDGES for d in (0, 1)]
    out = subprocess.run([str(tmp_path / "rule")], input="\n".join(" ".join(map(str, s)) for s in sizes),
                         capture_output=True, text=True, check=True).stdout.split()
    want = [x for *_, taken in EDGES for x in (taken, 1 - taken)]
    assert [int(x) for x in out] == want
