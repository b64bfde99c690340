"""What the compiler makes of the products' large tiles (velox_amd/csrc/tiles_mfma.h), checked without a GPU."""
import os
import re
import subprocess

import pytest

from velox_amd.kernels import build


@pytest.mark.parametrize("source", ["gemm.hip", "routed.hip"])
def test_nothing_moves_an_accumulator_between_matrix_instructions(source, tmp_path):
    """The matrix instructions are assembly to the compiler, so it does not wait for one before it moves the register that the instruction
    still writes: between the first and the last of a kernel there must be no such move, no spilled register and no branch target but the loop's."""
    try:
        hipcc = build.find_hipcc()
    except build.BuildError:
        pytest.skip("no hipcc here")
    out = os.path.join(tmp_path, "out.s")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(build.SOURCE_DIR, source), "-o", out], check=True, capture_output=True)
    with open(out, encoding="utf-8") as handle:
        kernels = re.findall(r"^(_Z12tiles_kernel\w+):(.*?)\.Lfunc_end", handle.read(), re.S | re.M)
    assert kernels
    for name, body in kernels:
        lines = body.splitlines()
        at = [i for i, line in enumerate(lines) if line.strip().startswith("v_mfma")]
        inside = [line.strip() for line in lines[at[0]:at[-1]]]
        assert not [line for line in inside if re.match(r"(v_accvgpr|scratch_|v_mov|\.LBB)", line)], name


def test_nor_in_the_kernel_that_holds_tiles_of_several_widths(tmp_path):
    """The plan's products choose between three such loops: each is one stretch of code without a branch target, with no move of an accumulator."""
    try:
        hipcc = build.find_hipcc()
    except build.BuildError:
        pytest.skip("no hipcc here")
    out = os.path.join(tmp_path, "out.s")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(build.SOURCE_DIR, "routed.hip"), "-o", out], check=True, capture_output=True)
    with open(out, encoding="utf-8") as handle:
        kernels = re.findall(r"^(_Z17plan_tiles_kernelILi(\d)\w+):(.*?)\.Lfunc_end", handle.read(), re.S | re.M)
    assert kernels
    for name, rows, body in kernels:
        counts = []
        for stretch in re.split(r"^\.LBB\w+:", body, flags=re.M):
            lines = [line.strip() for line in stretch.splitlines()]
            at = [i for i, line in enumerate(lines) if line.startswith("v_mfma")]
            if at:
                counts.append(len(at))
                assert not [line for line in lines[at[0]:at[-1]] if re.match(r"(v_accvgpr|scratch_|v_mov)", line)], name
        # two steps of 16 matrix instructions a pair of 32 x 32 tiles, at 2, 3 and 4 tiles of columns
        assert sorted(counts) == [16 * int(rows) * columns for columns in (2, 3, 4)], name
