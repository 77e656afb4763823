"""Vector registers of the kernels that one more register costs a wave.

The counts are read from the metadata of the library as built.  A SIMD holds
512 vector registers per lane: a kernel of 256 threads keeps w waves per SIMD
with at most 512 / w of them.
"""

import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _vgprs(tmp_path):
    from hipnufft import _build

    data = _build.LIB.read_bytes()
    out = {}
    for m in re.finditer(MAGIC, data):
        p = m.end()
        (n,) = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(n if n < 16 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx" not in name or not size:
                continue
            obj = tmp_path / "kernels.co"
            obj.write_bytes(data[m.start() + off:m.start() + off + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True,
                                   check=True).stdout
            for k in notes.split("- .agpr_count")[1:]:
                sym = re.search(r"\.name:\s+(\S+)", k)
                cnt = re.search(r"\.vgpr_count:\s+(\d+)", k)
                out[sym.group(1)] = int(cnt.group(1))
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    return {re.sub(r"\(anonymous namespace\)::|hn::|void ", "", n): v
            for n, v in zip(names, out.values())}


def test_waves(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    v = _vgprs(tmp_path)
    # adjoint last-axis pass of 300, 360, 600 and 720 points: 3 waves
    rows = [n for n in v if re.match(r"k_rows_adj<-?1, 12, (true|false), 0, 0>", n)]
    # stacked z axis of 64 to 128 points: 4 waves
    stack = [n for n in v if n.startswith("k_stack_adj<8, false>")]
    assert len(rows) == 4 and len(stack) == 1, sorted(v)
    assert all(v[n] <= 168 for n in rows), {n: v[n] for n in rows}
    assert all(v[n] <= 128 for n in stack), {n: v[n] for n in stack}
