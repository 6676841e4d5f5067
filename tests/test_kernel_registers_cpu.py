"""Registers and scratch of the built kernels where a change of a few decides
how many wavefronts a SIMD holds."""
import os
import re

import pytest

from tests.kernel_metadata import kernels

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tdvmc_amd", "libtdvmc.so")


@pytest.fixture(scope="module")
def built():
    return kernels(LIB)


def test_mixed_measurement_keeps_five_wavefronts(built):
    # 512 registers a SIMD, handed out in eights: five wavefronts have 96 each (3-D, 129 terms, N = 72, 1194 walkers:
    # 34 us with them, 40 with four)
    found = [(k, v) for k, v in built.items() if re.search(r"eval_kernel<float, \d, false, ", k)]
    assert len(found) == 12
    for name, v in found:
        # (two registers may spill: a coordinate read ahead, once stored and once loaded per walker)
        assert v["vgpr_count"] <= 96 and v["vgpr_spill_count"] <= 2, (name, v)


def test_mixed_observables_keep_eight_wavefronts(built):
    # one walker per workgroup (the form of few or large walkers, and of calls that ask for each walker's g(r)): the loop
    # over several walkers took 76 to 115 registers (N = 12, 192 walkers: 10.4 us without it, 13.4 with)
    found = [(k, v) for k, v in built.items() if re.search(r"obs_kernel<float, \d(, false)?>", k)]
    assert len(found) == 3
    for name, v in found:
        assert v["vgpr_count"] <= 64 and v["vgpr_spill_count"] == 0, (name, v)


def test_wide_spline_table_starts_at_lds_address_zero(built):
    # its rows' addresses are made by writing the row into byte 1 (kernels_sweep.hip): static LDS would come first
    found = [(k, v) for k, v in built.items() if re.search(r"sweep_kernel<float, \d, \d+, \d, true, false, true>", k)]
    assert len(found) == 72
    for name, v in found:
        assert v["group_segment_fixed_size"] == 0, (name, v)
