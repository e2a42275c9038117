"""The order in which the gradient kernels deal rows to the XCDs (`trl_amd/csrc/xcd_order.hpp`), in a host build of it."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "trl_amd", "csrc")

# One line per problem: total, wanted run -> run, workgroups, pieces dealt exactly once, fewest and most pieces of an XCD.
_SOURCE = r"""
#include "xcd_order.hpp"
#include <stdio.h>
#include <vector>
int main() {
    long long total, want, period;
    while (scanf("%lld %lld %lld", &total, &want, &period) == 3) {
        const unsigned run = trlk::xcd_run(total, want, period), grid = trlk::xcd_grid(total, run);
        std::vector<int> seen(total, 0);
        long long of_xcd[8] = {0}, once = 0, least = total, most = 0;
        for (unsigned w = 0; w < grid; ++w) {
            const int64_t p = trlk::xcd_piece(w, run);
            if (p < total) ++seen[p], ++of_xcd[w & 7];
        }
        for (int s : seen) once += s == 1;
        for (long long n : of_xcd) {
            least = n < least ? n : least;
            most = n > most ? n : most;
        }
        printf("%u %u %lld %lld %lld\n", run, grid, once, least, most);
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_rows_are_dealt_evenly_in_ten_runs_or_more(tmp_path):
    """Every piece once; at least 10 runs per XCD wherever runs are longer than one piece; and rounds of equal length: what the last
    round lacks is less than a piece of each run, so no XCD has a whole run more than another."""
    (tmp_path / "order.cpp").write_text(_SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(tmp_path / "order.cpp"), "-o", str(tmp_path / "order")], check=True)
    problems = [(n_seq * rows, want, rows)
                for n_seq in (1, 2, 3, 4, 6, 8, 10, 12, 16, 20, 31, 32, 64)
                for rows in (1, 7, 64, 137, 257, 300, 510, 586, 601, 1025, 2048)
                for want in (0, 1, 2, 12, 20, 24, 33, 83, 125, 157, 196)]
    out = subprocess.run([str(tmp_path / "order")], input="\n".join("%d %d %d" % p for p in problems), capture_output=True, text=True,
                         check=True, timeout=120).stdout.split("\n")
    for (total, want, rows), line in zip(problems, out):
        run, grid, once, least, most = map(int, line.split())
        rounds = grid // (8 * run)
        assert grid == 8 * run * rounds and once == total, (total, want, rows)
        assert run == 1 or total >= 80 * run - 8 * rounds and rounds >= 10, (total, want, rows, run, rounds)
        assert grid - total < 8 * rounds, (total, want, rows, run, rounds)
        assert most - least <= max(run, rounds), (total, want, rows, run, least, most)
