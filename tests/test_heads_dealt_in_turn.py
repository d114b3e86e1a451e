"""How the heads of a grid are dealt out (make_deal and deal of csrc/sma_internal.h, compiled for the host): about as many in turn as an XCD holds at once, whatever
divisors its share has, no group on two XCDs, every tile of every head once, and one head after the other where nothing is alike, the grid is one round
or the number of compute units is not known."""
import os
import shutil
import subprocess

import pytest

import _capi

CSRC = os.path.join(os.path.dirname(_capi.LIB), "csrc")

PROGRAM = r"""
#include "sma_internal.h"
#include <cstdio>
#include <vector>
int main()
{
    int heads, tiles, alike;
    long long resident;
    while (scanf("%d %d %lld %d", &heads, &tiles, &resident, &alike) == 4) {
        const sma::Deal d = sma::make_deal(alike != 0, heads, tiles, resident);
        std::vector<char> seen((size_t)heads * tiles);
        int ok = 1;
        for (int n = 0; n < heads * tiles; ++n) {
            const sma::Dealt w = sma::deal(d, tiles, n);
            if (w.head < 0 || w.head >= heads || w.tile < 0 || w.tile >= tiles) { ok = 0; break; }
            char &s = seen[(size_t)w.head * tiles + w.tile];
            if (s++) ok = 0;
            // the eighths of the grid are the XCDs' shares (heads that are a multiple of 8)
            if (d.together > 1 && n / (heads * tiles / 8) != w.head / (heads / 8)) ok = 0;
        }
        printf("%d %d\n", d.together, ok);
    }
}
"""


def _deals(tmp_path, grids):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no g++")
    (tmp_path / "deal.cpp").write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__=1", "-Wno-deprecated-declarations", f"-I{CSRC}",
                    f"-I{os.environ.get('ROCM_PATH', '/opt/rocm')}/include", str(tmp_path / "deal.cpp"), "-o", str(tmp_path / "deal")], check=True)
    text = "".join(f"{h} {t} {r} {int(a)}\n" for h, t, r, a in grids)
    out = subprocess.run([str(tmp_path / "deal")], input=text, capture_output=True, text=True, check=True).stdout.split()
    return [(int(g), ok == "1") for g, ok in zip(out[::2], out[1::2])]


def test_groups(tmp_path):
    grids = [(8 * share, tiles, resident, True)
             for share in list(range(1, 33)) + [61, 96, 97, 127] for tiles in (1, 2, 3, 4, 5, 7, 8, 16, 21, 26, 32, 33, 64) for resident in (256, 512, 768, 1024)]
    some = 0
    for (heads, tiles, resident, _), (g, ok) in zip(grids, _deals(tmp_path, grids)):
        share, holds = heads // 8, -(-(resident // 8) // tiles)
        assert ok and share % g == 0, (heads, tiles, resident, g)
        if heads * tiles <= resident:
            assert g == 1
            continue
        divisors = [x for x in range(1, share + 1) if share % x == 0]
        most = max(x for x in divisors if x <= holds)
        if 2 * most <= min(holds, share):                        # nothing near below it: at most two thirds above
            most = min([x for x in divisors if holds < x <= holds * 5 / 3], default=most)
        assert g == most <= holds * 5 / 3, (heads, tiles, resident, g)
        some += g > 1
    assert some > 500


def test_one_head_after_the_other(tmp_path):
    grids = [(192, 8, 768, False), (190, 8, 768, True), (192, 4, 768, True), (192, 8, 0, True), (8, 8, 0, True),
             (232, 32, 768, True), (1016, 4, 768, True)]                     # 29 and 127 heads a share, of which 3 and 24 are held at once
    assert _deals(tmp_path, grids) == [(1, True)] * len(grids)
    assert _deals(tmp_path, [(192, 8, 768, True), (192, 4, 512, True), (128, 32, 512, True), (104, 8, 512, True)]) == [
        (12, True), (12, True), (2, True), (13, True)]
