"""CPU restatement of csrc/attn_fwd.hip's requests for two tiles' mask bytes at once at any length (issue_mask_pair with FETCH = 2
and mask_words with pair_half): for every lane of every wavefront and every pair each 16-byte copy lies inside the mask and its
lane offset is a non-negative 32-bit number, and the chunks a lane converts hold the columns they stand for (the one in
which the row ends after the right shift that the kernel applies)."""
import numpy as np
import pytest

BM, BN = 128, 64


def _check(N):
    T, qtiles = (N + BN - 1) // BN, (N + BM - 1) // BM
    lane = np.arange(64)
    for qt in {0, qtiles - 1}:
        for wave in range(4):
            row_base = qt * BM + wave * 32
            for p in {0, (T - 1) // 2 - 1, (T - 1) // 2} - {-1}:
                held = np.full((32, 8), -1, dtype=np.int64)           # [row][position] -> first column
                chunk = ((lane & 7) ^ (lane >> 4)) << 4
                voff0 = (row_base + (lane >> 3)).astype(np.int64) * N + chunk
                vo = [voff0, voff0 + 64 - 2 * (chunk & 64)] * 2
                src, step, row_end = p * 2 * BN, 8 * N, N - p * 2 * BN
                grow = [row_base + 8 * j + (lane >> 3) for j in range(4)]
                if row_base + 32 > N:
                    step = 0
                    grow = [np.where(r < N, r, N - 1) for r in grow]
                    vo = [grow[j].astype(np.int64) * N + (chunk ^ (64 * (j & 1))) for j in range(4)]
                back = 0
                if row_end < 2 * BN:
                    back = 16 if p > 0 else 0
                    for j in range(4):
                        end = (chunk ^ (64 * (j & 1))) + 16
                        vo[j] = vo[j] + back - np.where(end > row_end, end - row_end, 0)
                for j in range(4):
                    assert (vo[j] >= 0).all() and (vo[j] < 2 ** 32).all(), (N, p, j)
                    base = src - back + j * step
                    assert base >= 0
                    addr = base + vo[j]
                    assert (addr >= 0).all() and (addr + 16 <= N * N).all(), (N, p, j)
                    dst = j * 1024 + lane * 16                          # byte in the wavefront's 4 KiB
                    assert ((dst >> 7) == 8 * j + (lane >> 3)).all()
                    held[dst >> 7, (dst >> 4) & 7] = addr - grow[j].astype(np.int64) * N
                for half in range(2):
                    x = 2 * p + half
                    if x >= T:
                        continue
                    end = N - x * BN
                    for l32 in range(32):
                        for c in range(4):                             # the tile's chunks: 2 hh and 2 hh + 1 of each lane half
                            col = held[l32, (4 * half + c) ^ ((l32 >> 1) & 7)]
                            want = x * BN + 16 * c
                            if want + 16 <= N:
                                assert col == want, (N, x, l32, c)
                            elif want < N:
                                assert c == end >> 4 and col + ((16 - (end & 15)) & 15) == want, (N, x, l32, c)


def test_every_length_up_to_700():
    for N in range(16, 701):
        _check(N)


@pytest.mark.parametrize("N", [1000, 1001, 2047, 4095, 8191, 46340])
def test_long_rows(N):
    _check(N)
