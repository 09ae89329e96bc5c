"""Registers of the built kernels, from the library's own metadata: what a
dispatch rule counts on about workgroups sharing a CU."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from hi_amd import _build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _kernels():
    """{kernel symbol: {metadata key: number}} of every gfx950 code object in libhi_rocm.so."""
    if not os.path.exists(_build.LIB):
        _build.build()
    data = open(_build.LIB, "rb").read()
    found = {}
    for m in re.finditer(MAGIC, data):
        base = m.start()
        n, at = struct.unpack_from("<Q", data, base + len(MAGIC))[0], base + len(MAGIC) + 8
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + tl]
            at += 24 + tl
            if not triple.endswith(b"gfx950") or size == 0:
                continue
            with tempfile.NamedTemporaryFile(suffix=".co") as f:
                f.write(data[base + off:base + off + size])
                f.flush()
                notes = subprocess.run([READELF, "--notes", f.name], capture_output=True, text=True, check=True).stdout
            for block in re.split(r"\n  - \.ag", notes)[1:]:
                block = ".ag" + block
                name = re.search(r"\.name: +(\S+)", block).group(1)
                found[name] = {k: int(v) for k, v in re.findall(r"\.(\w+_count|private_segment_fixed_size): +(\d+)", block)}
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_fused_kernel_two_workgroups_a_cu():
    """select_finish_kernel (four waves a workgroup) is launched with up to
    two workgroups a CU: at most 256 of a SIMD's 512 registers a wave (the
    metadata's VGPR count holds the AGPRs too), and no private memory."""
    k = {n: v for n, v in _kernels().items() if "select_finish_kernel" in n}
    assert len(k) == 8
    for name, v in k.items():
        assert v["vgpr_count"] <= 256, (name, v)
        assert v["private_segment_fixed_size"] == 0, (name, v)
