"""The FP64 sweep's launch rules on the host (tests/cpp/sweep_rules_check.cpp):
no lane of a walker without particles or k-space terms of its own where fewer
lanes would do, at most four k-space terms per lane while more lanes are to be
had, and phase tables only where a lane has more than one term to use them."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CHECK = os.path.join(HERE, "cpp", "build", "sweep_rules_check")


def _rules(rows):
    out = subprocess.run([CHECK], input="\n".join(" ".join(map(str, r)) for r in rows), capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


def _grid(D):
    # kmax of a shell of Kh pairs of vectors in D dimensions
    return [(D, N, 24, Kh, max(1, round((2 * Kh) ** (1.0 / D) / 2)) if Kh else 0, W) for N in (2, 5, 9, 15, 16, 17, 24, 31, 32, 33, 64, 100, 343)
            for Kh in (0, 1, 8, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257) for W in (1, 300, 1100, 2600, 3500, 7000, 20000, 100000)]


@pytest.mark.parametrize("D", [1, 2, 3])
def test_no_idle_lanes_and_few_terms_each(D):
    rows = _grid(D)
    got = _rules(rows)
    assert len(got) == len(rows)
    for (D, N, Ps, Kh, kmax, W), (lanes, table, lds) in zip(rows, got):
        assert lanes in (16, 32, 64) and lds <= 160 * 1024
        where = (D, N, Kh, W, lanes, table)
        # N = 9, 16 k, 3500 walkers: 18 us with 16 lanes, 25 with 64
        assert lanes == 16 or lanes // 2 < max(N, Kh), where
        # N = 8, 104 terms, 12331 walkers: 62 us with 32 lanes, 116 with 16
        assert lanes == 64 or Kh <= 4 * lanes, where
        # N = 12, 10 terms, 3256 walkers, 16 lanes: 15 us without tables, 19 with
        assert not table or Kh > lanes, where


def test_lanes_fill_the_chip():
    # 64: three wavefronts for every two SIMDs are there with fewer lanes
    for (lanes, _, _), want in zip(_rules([(3, 64, 32, 0, 0, W) for W in (500, 1535, 1536, 3071, 3072, 6143, 6144, 16384)]),
                                   (64, 64, 64, 64, 32, 32, 16, 16)):
        assert lanes == want
