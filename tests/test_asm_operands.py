"""Register operands of inline assembly, read off the gfx950 assembly hipcc makes of a probe kernel."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "threedgaussiansplatting.jl_amd", "csrc")
PROBE = """
#include "wave_sum.hpp"
__global__ void probe(const float* in, float* out) {
    float x[8], y[8];
    for (int k = 0; k < 8; ++k) x[k] = y[k] = in[64 * k + threadIdx.x];   // one value, two operands
    tdgs::halve_dpp<%d>(x, y);
    for (int k = 0; k < 8; ++k) out[64 * k + threadIdx.x] = x[k];
}
"""


@pytest.mark.parametrize("distance", [8, 4])
def test_halving_of_equal_values_keeps_their_registers_apart(distance, tmp_path):
    """halve_dpp writes its sums before it reads its second operands: none may share a register, also
    where the compiler knows both to hold the same value."""
    from tdgs_amd import build
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE % distance)
    subprocess.run([build.hipcc(), *build._flags(), "-S", "--cuda-device-only", str(src), "-o", str(asm)], check=True,
                   capture_output=True)
    adds = re.findall(r"v_add_f32_dpp (v\d+), (v\d+), (v\d+) row_ror", asm.read_text())
    assert len(adds) == 16
    first, second = adds[:8], adds[8:]   # x += x's partner, then x = y + y's partner in the other lanes
    assert all(d == a == b for d, a, b in first) and all(a == b for _, a, b in second)
    written = {d for d, _, _ in first}
    assert len(written) == 8 and written == {d for d, _, _ in second}
    assert not written & {a for _, a, _ in second}
