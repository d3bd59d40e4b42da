"""Host-side rules of the library, compiled from its own headers with the host compiler and run on the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tessera_amd" / "csrc"


def _run(tmp_path, source, *args):
    """Compiles one program against the library's headers and returns what it printed."""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True, timeout=60).stdout


def test_few_row_offsets_stay_in_32_bits(tmp_path):
    """Few-row products off the 16-byte grid: wherever the rule admits one, the largest offsets that the kernel's
    lanes form lie inside the buffer range (A) and inside 32 bits (B); ordinary sizes are admitted."""
    cases = _few_row_cases()
    out = _run(tmp_path, r"""
#include "few_rows.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  for (int i = 1; i + 4 < argc; i += 5)
    std::printf("%d\n", tsr950::few_rows16_in_range(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), atol(argv[i + 3]), atol(argv[i + 4])));
}
""", *[x for c in cases for x in c])
    got = [bool(int(x)) for x in out.split()]
    assert len(got) == len(cases)
    for (m, n, k, lda, ldb), ok in zip(cases, got):
        pitch = max(lda, -(-k // 8) * 8)
        # lane (row m - 1, upper half) of A's second load in a slice; row 31 and the last column of B's slice
        a_last = (m - 1) * pitch * 2 + 16 + 32 + 15
        b_last = (31 * ldb + n - 1) * 2 + 1
        assert not ok or (a_last < 2 ** 31 - 1 and b_last < 2 ** 32), (m, n, k)
        if max(lda, k) <= 1 << 24 and ldb <= 1 << 25:
            assert ok, (m, n, k)                          # nothing of the ordinary range is turned away
    assert not got[0] and not got[1] and got[2]


def _few_row_cases():
    cases = [(64, 8, 17_100_000), (1, 1 << 26, 32), (64, 50257, 4100)]
    cases += [(m, n, k) for m in (1, 2, 9, 32, 33, 64) for n in (8, 9, 1003, 1 << 24, 69_273_000, 69_274_000, 1 << 28)
              for k in (1, 33, 4097, 1 << 24, 17_043_000, 17_044_000, 34_600_000, 1 << 30, 2 ** 31 - 1)]
    return [(m, n, k, k, n) for m, n, k in cases] + [(3, 100, 64, 1 << 29, 104), (3, 100, 64, 64, 1 << 27)]
