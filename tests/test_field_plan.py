"""The field histogram's host tables fit the workspace its caller is asked for.

The tables are plain C++ (maxibone_amd/csrc/mxb_field_plan.h): a small program
plans calls over long, flat, uneven and ordinary extents, in bins of either
form, and compares the words in use with mxb_histogram_workspace_bytes' size.
"""
import os
import subprocess

from maxibone_amd import capi

CSRC = os.path.join(capi.PKG, "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "mxb_field_plan.h"
int main() {
    long long nz, ny, nx, fz, fy, fx, fb, vb;
    int mono;
    while (std::scanf("%lld %lld %lld %lld %lld %lld %lld %lld %d", &nz, &ny, &nx, &fz, &fy, &fx, &fb, &vb, &mono) == 9) {
        const int64_t n[3] = {nz, ny, nx}, nf[3] = {fz, fy, fx};
        mxb::FieldPlan p;
        mxb::make_field_plan(n, nf, fb, vb, mono != 0, p);
        std::printf("%lld %lld %d\n", (long long)(4 * p.table_words()),
                    (long long)mxb::field_workspace_bytes(nz, ny, nx), p.grouped ? 1 : 0);
    }
}
"""

LONG = [(1, 1, 140000), (2, 8, 200000), (200000, 3, 2), (3, 131200, 1), (70000, 70000, 2), (1, 1, 131133), (1, 1, 1 << 20)]
GRID = [(1, 1, 1), (13000, 13000, 13000), (40000, 1, 1), (8192, 8192, 8192), (4000, 50, 30000), (1024, 1024, 1024),
        (301, 257, 263), (39998, 1, 1), (8192, 16384, 8192)]


def test_field_tables_fit_the_workspace(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover",
                    "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    calls = []
    for n in LONG + GRID:
        for num, den in ((1, 1), (1, 2), (1, 3), (2, 3), (3, 2), (1, 9)):
            nf = tuple(max(1, e * num // den) for e in n)
            for fb, vb in ((1, 1), (2048, 4096), (2048, 32768), (2047, 16), (1 << 20, 32), (2, 40000)):
                calls += [(*n, *nf, fb, vb, 1), (*n, *nf, fb, vb, 0)]
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in calls), text=True,
                         stdout=subprocess.PIPE, check=True).stdout.split("\n")
    L, forms = capi.lib(), set()
    for c, line in zip(calls, out):
        used, room, grouped = map(int, line.split())
        assert room == L.mxb_histogram_workspace_bytes(*c[:3])
        assert used <= room, c
        forms.add(grouped)
    assert forms == {0, 1}
