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
    long long resident, bytes;
    while (scanf("%d %d %lld %d %lld", &heads, &tiles, &resident, &alike, &bytes) == 5) {
        const sma::Deal d = sma::make_deal(alike != 0, heads, tiles, resident, bytes);
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
    text = "".join(f"{h} {t} {r} {int(a)} {b}\n" for h, t, r, a, b in grids)
    out = subprocess.run([str(tmp_path / "deal")], input=text, capture_output=True, text=True, check=True).stdout.split()
    return [(int(g), ok == "1") for g, ok in zip(out[::2], out[1::2])]


def _grid(heads, N, D, alike=True, cus=256):
    """The forward's: 128 rows a work-group, three of them on a CU up to head dim 64 and two beyond."""
    return heads, -(-N // 128), (3 if D <= 64 else 2) * cus, alike, 4 * N * D


def test_groups(tmp_path):
    grids = [(8 * share, tiles, resident, True, 4 * 128 * tiles * D)
             for share in list(range(1, 33)) + [61, 96, 97, 127] for tiles in (1, 2, 3, 4, 5, 7, 8, 16, 21, 26, 32, 33, 64) for resident in (256, 512, 768, 1024)
             for D in (32, 128)]
    some = 0
    for (heads, tiles, resident, _, head_bytes), (g, ok) in zip(grids, _deals(tmp_path, grids)):
        share, held = heads // 8, resident // 8 / tiles          # heads that an XCD holds at once
        assert ok and share % g == 0, (heads, tiles, resident, g)
        if heads * tiles <= resident:
            assert g == 1
            continue
        divisors = [x for x in range(1, share + 1) if share % x == 0]
        below = max([x for x in divisors if x <= held], default=1)
        above = min([x for x in divisors if x > below], default=below)
        take = above * tiles * 3 <= resident // 8 * 5 and (2 * below * tiles <= resident // 8 or above * head_bytes <= 4.5 * 2 ** 20)
        assert g == (above if take else below), (heads, tiles, resident, head_bytes, g)
        assert g == 1 or g * tiles * 3 <= resident // 8 * 5
        some += g > 1
    assert some > 500


def test_named_grids(tmp_path):
    want = [(_grid(192, 1024, 64), 12), (_grid(192, 512, 128), 12), (_grid(128, 4096, 128), 2),                  # as many as are held, or most of them
            (_grid(128, 4096, 64), 4), (_grid(192, 700, 64), 24), (_grid(192, 800, 128), 8),                     # the next above where K and V fit
            (_grid(104, 1024, 128), 13),                                                                         # ... or where there is nothing near below
            (_grid(232, 4096, 64), 1), (_grid(488, 2048, 64), 1), (_grid(1016, 512, 64), 1)]                     # 29, 61 and 127 heads a share
    want += [(g, 1) for g in (_grid(192, 1024, 64, alike=False), _grid(190, 1024, 64), _grid(192, 512, 64), _grid(192, 1024, 64, cus=0), _grid(8, 1024, 64, cus=0))]
    assert _deals(tmp_path, [g for g, _ in want]) == [(n, True) for _, n in want]
