"""The FP64 measurement's launch rules on the host
(tests/cpp/eval_rules_check.cpp): fewer than four wavefronts per walker only
where that leaves the chip as many of them as it can hold, the k-space gradient by
runs and the rho_k table only where they were measured to pay."""
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
    rows = [(D, N, Ps, Kh, W, pp, 1, 1) for N in (2, 5, 9, 20, 25, 32, 33, 48, 49, 64, 100, 101, 343) for Ps in (4, 12, 24, 48)
            for Kh in (0, 1, 8, 16, 32, 64, 65, 128, 200, 258) for W in (1, 500, 1023, 1024, 2047, 2048, 4099, 16384, 100000)]
    got = _rules(rows)
    assert len(got) == len(rows)
    fewer = 0
    for row, (waves, *rest) in zip(rows, got):
        lds = rest[:3]
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
    # 3200 walkers in a 2-D trap, 48 knots: 60 us with one, 48 with two; per-particle output 69, 58 and 48 with four
    ((2, 48, 48, 0, 3200, 0), 2),
    ((2, 48, 48, 0, 3200, 1), 4),
    ((2, 90, 24, 0, 2100, 0), 4),
    ((1, 70, 29, 5, 12357, 0), 2),
    # the sizes the fewer wavefronts were measured at
    ((2, 25, 12, 16, 4099, 0), 1),
    ((3, 64, 32, 0, 16384, 0), 2),
    ((1, 20, 16, 0, 1024, 0), 2),
])
def test_measured_sizes(row, waves):
    assert _rules([row + (1, 1)])[0][0] == waves


# D, N, knots, terms, runs, largest component; by runs with 1, 2, 4 wavefronts; the table with real and complex parameters
@pytest.mark.parametrize("D,N,P_s,Kh,nrun,kmax,runs,table", [
    (3, 14, 48, 206, 68, 4, (0, 0, 0), 0),          # 3-D: short runs, few particles
    (3, 5, 24, 101, 41, 3, (0, 0, 0), 0),
    (2, 25, 12, 16, 5, 3, (0, 0, 0), 0),            # few terms
    (2, 25, 8, 50, 11, 5, (1, 1, 1), 0),
    (1, 20, 8, 7, 1, 7, (0, 0, 0), 0),
    (1, 20, 8, 11, 1, 11, (1, 0, 0), 0),
    (1, 108, 47, 40, 1, 40, (1, 1, 1), 0),
    (3, 180, 12, 3, 3, 1, (0, 0, 0), 1),
    (1, 20, 8, 24, 1, 24, (1, 1, 0), 0),
    (3, 33, 24, 32, 18, 2, (1, 1, 0), 0),
    (3, 47, 24, 128, 47, 4, (1, 1, 1), 0),
    (3, 48, 24, 128, 47, 4, (1, 1, 1), 1),
    (2, 400, 48, 258, 25, 12, (1, 1, 1), 1),
    (3, 343, 40, 128, 47, 4, (1, 1, 1), 1),
    (2, 86, 8, 64, 13, 6, (1, 1, 1), 0),            # little LDS: a few particles a pass
])
def test_forms_of_the_k_space_terms(D, N, P_s, Kh, nrun, kmax, runs, table):
    out = _rules([(D, N, P_s, Kh, 1000, 0, nrun, kmax)])[0][4:]
    assert (out[0], out[3], out[6]) == runs
    for real, cplx in ((out[7], out[8]),):          # four wavefronts
        assert (real > 0) == (table > 0) and (cplx > 0) == (table > 0)
        assert real == 0 or min(real, cplx) * 8 >= min(N, 64)
