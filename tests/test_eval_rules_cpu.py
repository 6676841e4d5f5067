"""The FP64 measurement's launch rules on the host
(tests/cpp/eval_rules_check.cpp): fewer than four wavefronts per walker only
where that leaves the chip as many of them as it can hold."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CHECK = os.path.join(HERE, "cpp", "build", "eval_rules_check")


def _rules(rows):
    out = subprocess.run([CHECK], input="\n".join(" ".join(map(str, r)) for r in rows), capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


@pytest.mark.parametrize("pp", [0, 1])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_fewer_wavefronts_leave_the_chip_full(D, pp):
    rows = [(D, N, Ps, Kh, W, pp) for N in (2, 5, 9, 20, 25, 32, 33, 48, 49, 64, 100, 101, 343) for Ps in (4, 12, 24, 48)
            for Kh in (0, 1, 8, 16, 32, 64, 65, 128, 200, 258) for W in (1, 500, 1023, 1024, 2047, 2048, 4099, 16384, 100000)]
    got = _rules(rows)
    assert len(got) == len(rows)
    fewer = 0
    for row, (waves, *lds) in zip(rows, got):
        assert waves in (1, 2, 4)
        if waves == 4:
            continue
        fewer += 1
        # wavefronts of a CU by LDS (four a workgroup): at least 12 of the 16 that the registers allow
        assert 4 * (160 * 1024 // lds[waves // 2]) >= 12, (row, waves, lds)
        # two for every SIMD of the chip's 1024
        assert row[4] * waves >= 2048, (row, waves)
    assert fewer > 100


@pytest.mark.parametrize("row,waves", [
    # 1328 walkers, 206 terms, complex parameters: 63 us with four, 158 with one
    ((3, 14, 48, 206, 1328, 0), 4),
    ((3, 5, 48, 257, 5915, 0), 4),
    # 588 walkers, 101 terms: 25 us with four, 32 with two
    ((3, 19, 24, 101, 588, 0), 4),
    # the sizes the fewer wavefronts were measured at
    ((2, 25, 12, 16, 4099, 0), 1),
    ((3, 64, 32, 0, 16384, 0), 2),
    ((1, 20, 16, 0, 1024, 0), 2),
])
def test_measured_sizes(row, waves):
    assert _rules([row])[0][0] == waves
