"""The steps a wave of the batched GEMV on the f32 matrix core takes
(csrc/dsv4_batch_walk.h, compiled here with g++): every chunk group that lies
in the row comes once, in order, and the scale-table entry that the wave reads
with each step -- and with the one past its last, which it reads too -- lies
inside the table that the launch sizes, L / 4 times nch entries per wave. CPU
only: an index past the table would be a read past the workgroup's LDS."""
import os
import shutil
import subprocess

import pytest

import common

CSRC = os.path.join(common.ROOT, "deepseek-v4-in-c_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "dsv4_batch_walk.h"

int main()
{
    long walks = 0;
    const int tcs[] = {4, 8, 16, 32, 64, 128, 192, 256};
    for (int tc : tcs)
        for (int nch = 1; nch <= 8; nch++)
            for (int ch = (nch - 1) * tc + 1; ch <= nch * tc; ch++)
                for (int L = 4; L <= 64 && L <= tc; L *= 2)
                    for (int j0 = 0; j0 < tc; j0 += L) {
                        const int groups = (L >> 2) * nch, steps = mf_steps(j0, L, tc, ch, nch);
                        MfWalk w(j0);
                        int s = 0;
                        walks++;
                        for (int u = 0; u < L >> 2; u++)
                            for (int n = 0; n < nch; n++) {
                                const int c = j0 + 4 * u + n * tc;
                                if (c >= ch) continue;
                                if (w.u != u || w.n != n || w.c != c ||
                                    w.entry(nch, groups) != u * nch + n) {
                                    printf("step %d: tc %d ch %d L %d j0 %d\n", s, tc, ch, L, j0);
                                    return 1;
                                }
                                w.next(j0, tc, ch);
                                s++;
                            }
                        const int e = w.entry(nch, groups);
                        if (s != steps || e < 0 || e >= groups) {
                            printf("%d of %d steps, then entry %d of %d: tc %d ch %d L %d j0 %d\n",
                                   s, steps, e, groups, tc, ch, L, j0);
                            return 1;
                        }
                    }
    printf("%ld walks\n", walks);
    return 0;
}
"""


def test_walk_stays_in_its_table(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    src = tmp_path / "walk.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "walk"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
