"""The built library's kernels keep their values in registers (the code objects'
own metadata; no GPU needed)."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from ainfer_amd._build import HIPCC, LIB

READELF = Path(HIPCC).resolve().parent.parent / "llvm" / "bin" / "llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """The device code objects of every offload bundle in the library."""
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            ident = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in ident and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 24)


def spills(tmp_path):
    """{kernel symbol: spilled vector registers}"""
    out = {}
    for i, co in enumerate(code_objects(LIB.read_bytes())):
        f = tmp_path / f"{i}.co"
        f.write_bytes(co)
        notes = subprocess.run([str(READELF), "--notes", str(f)], capture_output=True, text=True,
                               check=True).stdout
        for m in re.finditer(r"\.symbol:\s+(\S+)\.kd\b.*?\.vgpr_spill_count:\s+(\d+)", notes, re.S):
            out[m.group(1)] = int(m.group(2))
    return out


def test_no_kernel_spills(tmp_path):
    """All but the persistent stack, whose phases share one register budget."""
    if not LIB.exists() or not READELF.exists():
        pytest.skip("library or llvm-readelf missing")
    found = spills(tmp_path)
    assert sum("k_select" in k for k in found) == 40  # 5 expert counts x 4 widths x 2 forms
    assert not {k: n for k, n in found.items() if n and "k_decode_stack" not in k}
