"""Private memory of the built kernels (from the metadata of the gfx950 code
objects in the library): the FP32 lane-group spectral solve of up to 32 and
of 49 to 64 levels keeps its rows in registers, none of them in scratch, and
so do the FFT kernels for radices up to 20 in both precisions.  The fixed-point
spreading stays within 128 registers where its LDS lets four workgroups onto a
CU (records of up to 153 words)."""
import os
import re
import struct
import subprocess

import pytest

from doublyperiodicstokes_amd import build as b

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 ELF images of every offload bundle in the library."""
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + tl]
            p += 24 + tl
            if b"gfx950" in triple and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel name: (scratch bytes per lane, vector registers)}."""
    llvm = os.path.join(b.ROCM, "llvm", "bin")
    tool = os.path.join(llvm, "llvm-readelf")
    if not os.path.exists(b.lib_path()):
        b.build()
    if not os.path.exists(tool):
        pytest.skip("llvm-readelf not found")
    d = tmp_path_factory.mktemp("co")
    out = {}
    with open(b.lib_path(), "rb") as f:
        data = f.read()
    for i, image in enumerate(code_objects(data)):
        path = d / ("%d.co" % i)
        path.write_bytes(image)
        text = subprocess.run([tool, "--notes", str(path)], stdout=subprocess.PIPE, check=True).stdout.decode()
        for block in text.split("- .agpr_count:")[1:]:
            get = lambda key: re.search(r"\.%s:\s+(\S+)" % key, block).group(1)  # noqa: E731
            out[get("name")] = int(get("private_segment_fixed_size")), int(get("vgpr_count"))
    return out


@pytest.mark.parametrize("lpm,e", [(8, 2), (16, 2), (16, 4)])
def test_lane_group_solve_has_no_scratch(kernels, lpm, e):
    found = [v for k, v in kernels.items() if "k_spectralIfLi%dELi%dE" % (lpm, e) in k]
    assert len(found) == 1
    assert found[0][0] == 0


@pytest.mark.parametrize("real", ["f", "d"])
@pytest.mark.parametrize("rmax", [10, 16, 20])
def test_fft_kernels_have_no_scratch(kernels, real, rmax):
    for name in ("k_fft_colsI%sLi%dELin1E", "k_fft_colsI%sLi%dELi1E", "k_fft_rows_fwdI%sLi%dE", "k_fft_rows_invI%sLi%dE"):
        found = [v[0] for k, v in kernels.items() if name % (real, rmax) in k]
        assert found == [0], name


@pytest.mark.parametrize("words", [8, 10])
def test_fixed_point_spreading_registers(kernels, words):
    found = [v for k, v in kernels.items() if "k_spread_fxILi%dE" % words in k]
    assert found and all(scratch == 0 and vgpr <= 128 for scratch, vgpr in found)
