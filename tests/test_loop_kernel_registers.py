"""Registers of the solve-loop kernels on symmetric diagonals, from the
compiler's resource remarks (cgxx_amd/lib/kernel_resources.json).

A kernel whose grid fills the chip many times over keeps 8 waves per SIMD: at
most 64 VGPRs.  Three have fewer waves than that to run: the step of the loop
of two kernels (at most 1,024 blocks of 4 waves) and the two dots with four rows
per thread (at most 4,096 blocks of one wave).  On 256 compute units of 4 SIMDs
that is 4 waves per SIMD, so all of them are resident at once with up to
128 VGPRs, and the registers hold loads in flight instead.  None spills.
"""
import json
import re

import pytest

from cgxx_amd import build

LIMITS = {
    r"k_matvec_sym64<": 64, r"k_pcg_matvec_dot_sym64<": 64, r"k_pcg_update_small<": 64,
    r"k_poly_quad<": 64, r"k_pcg_step_sym64<": 128, r"k_poly_quad_dot<": 128,
    r"k_mp_matvec_dot_quad<": 128,
}


@pytest.mark.parametrize("pattern", sorted(LIMITS))
def test_registers(pattern):
    with open(build.RESOURCES) as f:
        found = {k: r for k, r in json.load(f).items() if re.search(pattern, k)}
    assert found
    for name, r in found.items():
        assert r["sgpr"] <= 80, (name, r)
        assert r["vgpr"] + r.get("agpr", 0) <= LIMITS[pattern], (name, r)
        assert r["scratch"] == 0, (name, r)
