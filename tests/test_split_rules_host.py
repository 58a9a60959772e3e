"""The rules that cut a call's keys into splits or ranges (csrc/decode_split.h), compiled for the
host: standard C++ without a device."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "modelcore_amd" / "csrc"

SPLIT_LEN = """
#include "decode_split.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char **argv) {
  long long v[6];
  for (int i = 1; i + 5 < argc; i += 6) {
    for (int j = 0; j < 6; ++j) v[j] = atoll(argv[i + j]);
    printf("%lld\\n", (long long)mcamd::split_len(v[0], v[1], v[2], v[3], v[4], v[5],
                                                  [](long long) { return true; }));
  }
}
"""


def _run(tmp_path, source, args):
    cxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/bin/amdclang++"
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", str(CSRC), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe), *[str(a) for a in args]], check=True, capture_output=True, text=True)
    return [int(x) for x in out.stdout.split()]


def _split_lens(tmp_path, cases):
    return _run(tmp_path, SPLIT_LEN, [x for c in cases for x in c])


def test_rows_shorter_than_their_cache_keep_their_decode_workgroups(tmp_path):
    """Splits longer than 256 keys only where the grid stays at 8192 workgroups or more: the length
    follows the cache's capacity, and rows that fill a part of it get that part of the grid."""
    rows = [1, 3, 8, 16, 32, 64]
    cases = [(b, h, d, t, w, e) for b in rows for h in (1, 4, 8, 12) for d in (16, 64, 96, 256)
             for t in (300, 2048, 8218, 16384, 65536, 131072) for w in (-1, 1500) for e in (2, 4)]
    for (b, h, d, t, w, e), n in zip(cases, _split_lens(tmp_path, cases)):
        span = min(t, w + 1) if w >= 0 else t
        assert n in (64, 128, 256, 512, 1024, 2048)
        if n > 256:
            assert b * h * -(-span // n) >= 8192, (b, h, d, t, w, e, n)
        # Rows of an eighth of the cache's length: a workgroup per compute unit, or 256 keys each.
        assert n <= 256 or b * h * -(-(span // 8) // n) >= 256, (b, h, d, t, w, e, n)


def test_short_caches_of_many_rows_are_not_cut(tmp_path):
    cases = [(b, h, 64, t, -1, 2) for b, h, t in ((300, 8, 512), (300, 8, 257), (255, 8, 512), (300, 8, 513),
                                                  (300, 8, 256))]
    assert _split_lens(tmp_path, cases) == [512, 512, 256, 256, 256]


@pytest.mark.parametrize("t_max", [(1 << 24) + 1, 135_000_000, 1 << 30])
def test_decode_splits_fit_a_grid(tmp_path, t_max):
    cases = [(b, h, 8, t_max, -1, e) for b in (1, 5, 64) for h in (1, 8) for e in (2, 4)]
    for n in _split_lens(tmp_path, cases):
        assert -(-t_max // n) <= 65535
