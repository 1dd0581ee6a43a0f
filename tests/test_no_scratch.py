"""No kernel of the built library spills registers to scratch memory, from the
metadata the compiler writes beside each kernel (no GPU needed)."""
from __future__ import annotations

import importlib
import os
import re
import struct
import subprocess
from pathlib import Path

from conftest import PKG  # noqa: F401

build = importlib.import_module("inference_systems_amd.build")

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib: Path):
    """The gfx950 code objects in the library, one per source file."""
    data = lib.read_bytes()
    for at in (m.start() for m in re.finditer(re.escape(MAGIC), data)):
        count, pos = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + length].decode()
            pos += 24 + length
            if build.ARCH in target and size:
                yield data[at + offset:at + offset + size]


def test_no_kernel_uses_scratch(tmp_path):
    readelf = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin" / "llvm-readelf"
    kernels = {}
    for i, obj in enumerate(_code_objects(build.LIB_PATH)):
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        notes = subprocess.run([str(readelf), "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for entry in notes.split("- .agpr_count:")[1:]:
            field = lambda key: re.search(rf"^\s*\.{key}:\s+(\S+)", entry, re.M).group(1)  # noqa: E731
            kernels[field("symbol")] = [int(field(k)) for k in ("private_segment_fixed_size", "vgpr_spill_count")]
    assert any("mfma_wide_kernel" in k for k in kernels) and any("splitk_decode_kernel" in k for k in kernels)
    spilling = {k: v for k, v in kernels.items() if any(v)}
    assert not spilling, f"{len(spilling)} of {len(kernels)} kernels (scratch bytes, spilled VGPRs): {spilling}"
