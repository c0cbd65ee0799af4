"""Registers of the kernels whose launch plans count on a number of waves to a compute unit, as the
compiler noted them in the library that was built."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cudarl-arena_amd", "lib", "libcrl.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: {field: number}} of the gfx950 code in the library."""
    data = open(LIB, "rb").read()
    at = data.index(MAGIC)
    (count,), pos = struct.unpack_from("<Q", data, at + len(MAGIC)), at + len(MAGIC) + 8
    for _ in range(count):
        offset, size, n = struct.unpack_from("<3Q", data, pos)
        target = data[pos + 24:pos + 24 + n].decode()
        pos += 24 + n
        if target.endswith("gfx950"):
            break
    else:
        pytest.fail("no gfx950 code in " + LIB)
    path = tmp_path_factory.mktemp("code") / "code.o"
    path.write_bytes(data[at + offset:at + offset + size])
    out, found = subprocess.check_output([READELF, "--notes", str(path)], text=True), {}
    for block in re.split(r"\n\s+- \.agpr_count", out)[1:]:
        name = re.search(r"\.name:\s+(_Z\S+)", block)
        found[name.group(1)] = {k: int(v) for k, v in re.findall(r"\.(vgpr_count|vgpr_spill_count|private_segment_fixed_size):\s+(\d+)", block)}
    return found


def test_lane_waves_to_a_simd(kernels):
    """plan_fused puts up to 24 lane waves on a compute unit, 20 with episode statistics or a budget (the
    third form): 512 / 6 and 512 / 5 registers, in eights."""
    lanes = {k: v for k, v in kernels.items() if "k_fused_lanes" in k}
    assert len(lanes) == 12
    for name, got in lanes.items():
        assert got["vgpr_count"] <= (96 if "ELi2EEE" in name else 80), (name, got)
        assert got["private_segment_fixed_size"] == 0 and got["vgpr_spill_count"] == 0, (name, got)


def test_waves_that_keep_rows(kernels):
    """Up to sixteen 64-env waves that keep rows in LDS to a compute unit: 512 / 4 registers, and nothing in scratch."""
    rows = {k: v for k, v in kernels.items() if re.search(r"k_fused_ticketsILi[48]ELi[012]ELb0ELb[01]ELi[1-9]EE", k)}
    assert len(rows) == 10
    for name, got in rows.items():
        assert got["vgpr_count"] <= 128, (name, got)
        assert got["private_segment_fixed_size"] == 0 and got["vgpr_spill_count"] == 0, (name, got)
