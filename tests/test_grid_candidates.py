"""Grid sizes the autotuners time for one schedule (grid_candidates in np_common.h): the rule, one, two
and all that fit, each once."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG_DIR

SOURCE = """
#include <cstdio>
#include "np_common.h"
int main() {
    for (int rule = 0; rule <= 6; ++rule)
        for (int occ = 1; occ <= 6; ++occ) {
            int w[4];
            const int k = np::grid_candidates(rule, occ, w);
            printf("%d %d", rule, occ);
            for (int i = 0; i < k; ++i) printf(" %d", w[i]);
            printf("\\n");
        }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_size_once_and_none_lost(tmp_path):
    (tmp_path / "g.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(PKG_DIR, "csrc"), str(tmp_path / "g.cpp"), "-o", str(tmp_path / "g")],
                   check=True, timeout=120)
    out = subprocess.run([str(tmp_path / "g")], check=True, stdout=subprocess.PIPE, text=True, timeout=20).stdout
    for line in out.splitlines():
        rule, occ, *got = (int(x) for x in line.split())
        assert got[0] == 0 and got[1:] == sorted({w for w in (1, 2, occ) if w <= occ and w != rule}), line
        # with what the rule takes, one, two and all that fit are timed
        assert {1, min(2, occ), occ} <= set(got) | {rule}, line
