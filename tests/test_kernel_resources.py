"""Resources of the built leaf kernels, from the code objects' own metadata
(host only): the whole-tile kernels of the spread loop, the ones an aligned
multiply runs on, keep everything in registers."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 code objects of every offload bundle in a library."""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if data[pos + 24:pos + 24 + n].endswith(b"gfx950"):
                yield data[at + off:at + off + size]
            pos += 24 + n
        at = data.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_whole_tile_leaf_kernels_use_no_scratch(tmp_path):
    with open(os.path.join(ROOT, "fast-matmul_amd", "fastmm", "libfastmm.so"), "rb") as f:
        data = f.read()
    scratch = {}
    for i, obj in enumerate(_code_objects(data)):
        if b"fm_gemm_kernel" not in obj:
            continue
        p = tmp_path / ("co%d" % i)
        p.write_bytes(obj)
        notes = subprocess.check_output([READELF, "--notes", str(p)], text=True)
        for kernel in notes.split("- .agpr_count")[1:]:
            name = re.search(r"\.name:\s*(\S+)", kernel).group(1)
            scratch[name] = int(re.search(r"\.private_segment_fixed_size:\s*(\d+)", kernel).group(1))
    # fm_gemm_kernel<T, BM, BN, BK, WM, WN, MINW, UNR, PIPE = 3 (spread), FULL = true, ANY = false>
    full = {n: b for n, b in scratch.items() if re.search(r"fm_gemm_kernelI[df](Li\d+E){7}Li3ELb1ELb0E", n)}
    # 128x128, 128x256, 128x64, 64x128, 64x64, 32x32 in both types, 128x96 in FP64
    assert len(full) >= 13
    assert not {n: b for n, b in full.items() if b}
