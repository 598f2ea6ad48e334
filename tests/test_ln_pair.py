"""The LayerNorm fold's row partials as two lanes share them (sh_ln_pair.h), enumerated in a host program: every request of
both lanes lies inside its row, and each partial pair is one lane's own exactly once, the lower lane's first."""
from __future__ import annotations

import subprocess

from conftest import ROOT

_MAIN = r"""
#include "sh_ln_pair.h"
#include <cstdio>
int main() {
    for (uint32_t parts = 2; parts <= 32; parts += 2) {          // the counts that are held in registers
        const uint32_t n = parts / 2, h0 = ln_pair_count(n, 0);
        if (h0 > 8 || h0 + ln_pair_count(n, 1) != n) { printf("parts %u: counts\n", parts); return 1; }
        uint32_t next = 0;
        for (uint32_t up = 0; up < 2; ++up)
            for (uint32_t h = 0; h < h0; ++h) {
                const uint32_t at = ln_pair_at(n, up, h);
                if (at >= n) { printf("parts %u lane %u request %u: entry %u of %u\n", parts, up, h, at, n); return 1; }
                if (h < ln_pair_count(n, up) && at != next++) { printf("parts %u: order\n", parts); return 1; }
            }
        if (next != n) { printf("parts %u: %u of %u entries\n", parts, next, n); return 1; }
    }
    return 0;
}
"""


def test_requests_stay_inside_the_row(tmp_path):
    src, exe = tmp_path / "pair.cpp", tmp_path / "pair"
    src.write_text(_MAIN)
    subprocess.run(["g++", "-O1", f"-I{ROOT}/softhier_mlir_amd/csrc", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
