"""What the compiler made of kernels whose speed rests on their values staying in registers:
the resource notes of the code objects inside the built library."""
import os
import re
import struct
import subprocess

import pytest

import zzref as Z

LIB = os.path.join(Z.ROOT, "zunzuncito_amd", "libzzmoe.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled kernel name: (scratch bytes a lane, LDS bytes)} of every gfx950 kernel."""
    with open(LIB, "rb") as f:
        lib = f.read()
    magic, found, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    obj = tmp_path_factory.mktemp("obj") / "code.o"
    while (at := lib.find(magic, at)) >= 0:
        n, pos = struct.unpack_from("<Q", lib, at + 24)[0], at + 32
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", lib, pos)
            if b"gfx950" in lib[pos + 24:pos + 24 + tl] and size:
                obj.write_bytes(lib[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                for k in notes.split("  - .agpr_count:")[1:]:
                    get = lambda f: re.search(r"\." + f + r":\s+(\S+)", k).group(1)
                    found[get("symbol")[:-3]] = int(get("private_segment_fixed_size")), int(get("group_segment_fixed_size"))
            pos += 24 + tl
        at += 24
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout
    return dict(zip((n.split("(")[0].removeprefix("void ") for n in names.splitlines()), found.values()))


def test_matmul_sums_in_registers(kernels):
    """No scratch, and no LDS beyond the four waves' partial sums (4 x 4 rows x 8 tokens)."""
    mm = {k: v for k, v in kernels.items() if k.startswith("zz_matmul_f32_kernel<")}
    assert len(mm) == 32
    assert not [(k, v) for k, v in mm.items() if v[0] or v[1] > 512]
