"""Register allocation of the inline assembly that composites a group's
samples (add_color, pyvr_amd/csrc/hvr_device.h): three multiply-adds in one
block, the first of which writes a colour while the inputs of the others are
still to be read.  Compiled to assembly for gfx950 with the library's flags,
in functions where an input holds the same value as an accumulator, so that
the compiler may give both one register unless the block forbids it.  Runs on
the CPU (nothing is executed)."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# accumulators C0..C2 and inputs tl, q0..q2 as parts of the loaded values
CASES = {
    "q1_is_c0": "float C0 = v[0], C1 = v[1], C2 = v[2], tl = v[3], q0 = v[4], q1 = v[0], q2 = v[5]",
    "q2_is_c0": "float C0 = v[0], C1 = v[1], C2 = v[2], tl = v[3], q0 = v[4], q1 = v[5], q2 = v[0]",
    "q2_is_c1": "float C0 = v[0], C1 = v[1], C2 = v[2], tl = v[3], q0 = v[4], q1 = v[5], q2 = v[1]",
    "tl_is_c0": "float C0 = v[0], C1 = v[1], C2 = v[2], tl = v[0], q0 = v[3], q1 = v[4], q2 = v[5]",
    "tl_is_c1": "float C0 = v[0], C1 = v[1], C2 = v[2], tl = v[1], q0 = v[3], q1 = v[4], q2 = v[5]",
}


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    """The fmac operands (dst, src0, src1) of every case's block."""
    from pyvr_amd import _build

    if shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("asm")
    src = d / "cases.hip"
    body = "".join(f'extern "C" __global__ void {name}(const float *p, float *o) {{\n'
                   "  float v[6];\n  for (int k = 0; k < 6; ++k) v[k] = p[64 * k + threadIdx.x];\n"
                   f"  {init};\n  add_color<2, 0>(tl, q0, q1, q2, C0, C1, C2);\n"
                   "  o[threadIdx.x] = C0; o[64 + threadIdx.x] = C1; o[128 + threadIdx.x] = C2;\n}\n"
                   for name, init in CASES.items())
    src.write_text('#include "hvr_device.h"\nusing namespace hvr;\n' + body)
    out = d / "cases.s"
    subprocess.run([_build.hipcc()] + _build.HIPCC_FLAGS +
                   ["-S", "--offload-device-only", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"), str(src), "-o", str(out)],
                   check=True, capture_output=True, text=True)
    text = out.read_text()
    res = {}
    for name in CASES:
        code = text[text.index(f"\n{name}:"):]
        code = code[:code.index("s_endpgm")]
        res[name] = re.findall(r"v_fmac_f32_dpp (v\d+), (v\d+), (v\d+) ", code)
    return res


@pytest.mark.parametrize("case", sorted(CASES))
def test_no_input_shares_a_register_written_before_it_is_read(blocks, case):
    fmacs = blocks[case]
    assert len(fmacs) == 3
    for k, (dst, _, _) in enumerate(fmacs):
        for _, a, b in fmacs[k + 1:]:
            assert dst not in (a, b), fmacs
