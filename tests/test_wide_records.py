"""The records of the 16-wide hierarchy (csrc/pg_wide.hpp), by g++: at every
number of points that a call takes they fit into the memory they are given, and
the subtree that starts last in any class has its record inside it."""
import os
import shutil
import subprocess

from tests import emu

PROGRAM = r"""
#include "pg_wide.hpp"
#include <stdio.h>
using namespace pg;
int main() {
    for (uint32_t n = 1; n <= (uint32_t)kMaxPoints; ++n) {
        if (!wide_fits(n)) { printf("%u points: %llu records\n", n, (unsigned long long)wide_records(n)); return 1; }
        const uint64_t records = wide_records(n);
        for (int k = 1; k <= wide_class(n); ++k)
            if (wide_slot(n, k, n - wide_least(k)) >= records) { printf("%u points, class %d\n", n, k); return 1; }
        if (n > 33 && wide_class(n) < wide_class(n - 1)) return 1;
    }
    printf("ok\n");
}
"""


def test_records_fit_at_every_size(tmp_path):
    src, prog = tmp_path / "fits.cpp", str(tmp_path / "fits")
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX") or shutil.which("g++"), "-std=c++17", "-O2", f"-I{emu.HERE}",
                    f"-I{emu.CSRC}", str(src), "-o", prog], check=True)
    r = subprocess.run([prog], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
