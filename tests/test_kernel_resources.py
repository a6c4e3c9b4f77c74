"""What the compiler gave the kernels of the built library: no kernel keeps registers in scratch memory, apart from the
head_dim-512 prefill's item loop. A spilled register is reloaded where it is used next, on a step's tail a memory
round trip on every workgroup's critical path, and every workgroup of the kernel is launched with scratch."""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parent.parent / "gemma4-webgpu_amd" / "lib" / "libg4attn.so"
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib: bytes):
    """The gfx950 ELF images of the library's offload bundles."""
    at = lib.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", lib, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", lib, p)
            name = lib[p + 24:p + 24 + length].decode()
            p += 24 + length
            if name.endswith("gfx950") and size:
                yield lib[at + offset:at + offset + size]
        at = lib.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> (scratch bytes a lane, spilled vector registers) from the code objects' metadata."""
    if not LIB.exists() or not Path(READELF).exists():
        pytest.skip("needs the built library and llvm-readelf")
    found = {}
    for i, image in enumerate(code_objects(LIB.read_bytes())):
        path = tmp_path_factory.mktemp("co") / f"{i}.co"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"\n  - \.a", notes)[1:]:
            value = lambda key: re.search(rf"\.{key}:\s+(\S+)", k)[1]  # noqa: E731
            found[value("symbol").removesuffix(".kd")] = int(value("private_segment_fixed_size")), int(value("vgpr_spill_count"))
    return found


def test_kernels_found(kernels):
    assert sum("k_attn_step" in k for k in kernels) >= 8 and len(kernels) > 80


def test_no_kernel_uses_scratch(kernels):
    scratch = {k: v for k, v in kernels.items() if v != (0, 0) and "k_prefill_pp512" not in k}
    assert not scratch, scratch
