"""The cut of a multihistogram run over workgroups, on the CPU: for every
number of bins (more blocks than compute units included), temperatures and runs
it ends, covers the bins once and stays within LDS."""
import pathlib
import shutil
import subprocess

import pytest

from conftest import PKG_DIR

PROG = """
#include <cstdio>
#include <cstdlib>
#include "ptmc_multihist_cut.hpp"
using namespace ptmc;

int main(int argc, char **argv)
{
    const int cus = atoi(argv[1]);
    const size_t max_lds = (size_t)atol(argv[2]);
    const int Rs[] = {1, 2, 8, 20, 32, 40, 48, 90, 94, 150, 300};
    const int runs[] = {1, 2, 3, 16, 255, 300};
    long bad = 0;
    auto check = [&](int R, size_t bins, int n) {
        const MhCut c = mh_cut(R, bins, n, cus, max_lds);
        const size_t slice = bins < (size_t)c.wg_blk * MH_BINS ? bins : (size_t)c.wg_blk * MH_BINS;
        const bool covers = c.n_wg >= 1 && c.wg_blk >= 1 && (size_t)c.n_blk * MH_BINS >= bins &&
                            (long)c.n_wg * c.wg_blk >= c.n_blk && (long)(c.n_wg - 1) * c.wg_blk < c.n_blk;
        const bool fits = c.keep ? c.lds == 8 * (mh_lds(R, true, false) + mh_slice(R, slice)) && c.lds <= max_lds
                                 : c.lds == 8 * mh_lds(R, false, false);
        // every slice fits once there are as many workgroups as compute units, or it is not kept
        const size_t most = (size_t)((c.n_blk + cus - 1) / cus) * MH_BINS, least = bins < most ? bins : most;
        const size_t base = 8 * mh_lds(R, true, false);
        const bool could = base < max_lds && 8 * mh_slice(R, least) <= max_lds - base;
        if (!covers || !fits || (c.n_wg > 1 && c.n_wg > cus) || could != c.keep) {
            if (bad++ < 5) std::printf("R %d bins %zu runs %d: n_wg %d wg_blk %d keep %d\\n", R, bins, n, c.n_wg, c.wg_blk, (int)c.keep);
        }
    };
    for (int R : Rs)
        for (int n : runs) {
            for (int nb = 1; nb <= 400; ++nb) check(R, (size_t)nb * nb, n);
            for (size_t bins = 1; bins < 1400; ++bins) check(R, bins, n);
            for (size_t bins : {(size_t)32768, (size_t)32769, (size_t)33152, (size_t)1 << 22, (size_t)1 << 26}) check(R, bins, n);
        }
    std::printf("%ld bad\\n", bad);
    return bad != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("cut")
    (d / "cut.cpp").write_text(PROG)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{pathlib.Path(PKG_DIR) / 'csrc'}", str(d / "cut.cpp"), "-o",
                    str(d / "cut")], check=True)
    return d / "cut"


# the MI355X, a device that shows a part of it, and a tenth of the LDS
@pytest.mark.parametrize("cus,lds", [(256, 163840), (80, 163840), (32, 163840), (256, 16384)])
def test_cut_ends_and_covers(program, cus, lds):
    p = subprocess.run([str(program), str(cus), str(lds)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
