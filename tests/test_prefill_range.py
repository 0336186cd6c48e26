"""The prefill kernel's key ranges and page-table indexes (csrc/kvrt_range.h,
compiled for the host) over every position of a chunk: a length below the query
count, which only graph replays reach, takes no key and reads no page entry."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "gemma-4-omni_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <algorithm>
#include "kvrt_range.h"
using namespace kvrt;
int main() {
    const int block = 32, shift = 4, pt_stride = 64;
    long n = 0, empty = 0;
    for (int base = -300; base <= 600; base += base < 40 ? 1 : 7)
        for (int qf = 0; qf < 260; qf += 1 + qf / 3)
            for (int ql : {qf, qf + 1, qf + 7, qf + 127})
                for (int window : {0, 1, 24, 200})
                    for (int nks : {1, 2, 3, 8, 16}) {
                        const int lo = window > 0 ? std::max(0, base + qf - window + 1) : 0, hi = base + ql + 1;
                        int covered = 0, at = lo;
                        for (int ks = 0; ks < nks; ++ks, ++n) {
                            const KeyRange r = prefill_range(base, qf, ql, window, nks, ks, block);
                            for (int parts : {1, 2, 4}) {
                                // the kernel's count of groups: it fetches where this is positive
                                const int groups = (r.kend - r.kstart + block * parts - 1) / (block * parts);
                                if ((groups > 0) != (r.kend > r.kstart)) return std::printf("groups %d of [%d, %d)\n", groups, r.kstart, r.kend), 1;
                                for (int p = 0; p < parts && groups > 0; ++p)
                                    for (int g = 0; g <= groups + 2; ++g) {
                                        const int t = r.kstart + (g * parts + p) * block, lp = std::min(t, r.kend - 1) >> shift;
                                        if (!page_in_table(lp, pt_stride)) return std::printf("page %d of [%d, %d)\n", lp, r.kstart, r.kend), 1;
                                    }
                            }
                            if (r.kend <= r.kstart) { ++empty; continue; }
                            if (r.kstart != at || r.kstart < 0) return std::printf("range starts at %d, not %d\n", r.kstart, at), 1;
                            covered += r.kend - r.kstart;
                            at = r.kend;
                        }
                        if (covered != std::max(0, hi - lo)) return std::printf("%d keys of [%d, %d)\n", covered, lo, hi), 1;
                    }
    if (page_in_table(-1, pt_stride) || page_in_table(pt_stride, pt_stride) || !page_in_table(0, 1)) return 1;
    return std::printf("%ld ranges, %ld empty\n", n, empty), empty == 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_ranges_cover_the_keys_and_stay_in_the_page_table(tmp_path):
    src = tmp_path / "range.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "range"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
