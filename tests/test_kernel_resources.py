"""Registers and LDS of the built kernels, from the metadata of the library's
own code objects: what a kernel's comment says fits a CU does fit it."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
READELF = os.path.join(LLVM, "llvm-readelf")
OBJCOPY = os.path.join(LLVM, "llvm-objcopy")
LDS_CU, LDS_GRANULE, VGPRS_LANE, VGPR_GRANULE = 160 * 1024, 1280, 512, 8


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: (LDS bytes, VGPRs)} of every kernel in the library."""
    from nest_splat import _lib
    if not (os.path.exists(READELF) and os.path.exists(OBJCOPY)):
        pytest.skip("the ROCm LLVM tools are not installed")
    d = tmp_path_factory.mktemp("co")
    so = shutil.copy(os.path.join(os.path.dirname(_lib.__file__), "libnest_splat.so"), d)
    fat = str(d / "fat")
    subprocess.run([OBJCOPY, f"--dump-section=.hip_fatbin={fat}", so, str(d / "out.so")], check=True, capture_output=True)
    blob = open(fat, "rb").read()
    found = {}
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", blob):
        at = m.end()
        (n,), at = struct.unpack_from("<Q", blob, at), at + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, at)
            ident, at = blob[at + 24:at + 24 + idlen], at + 24 + idlen
            if size == 0 or b"gfx950" not in ident:
                continue
            co = d / "co.elf"
            co.write_bytes(blob[m.start() + off:m.start() + off + size])
            notes = subprocess.run([READELF, "--notes", str(co)], check=True, capture_output=True, text=True).stdout
            for k in re.split(r"\n  - \.", notes)[1:]:
                name = re.search(r"\.name: +(_Z\w+)", k)
                if name:
                    found[name.group(1)] = (int(re.search(r"\.group_segment_fixed_size: +(\d+)", k).group(1)),
                                            int(re.search(r"\.vgpr_count: +(\d+)", k).group(1)))
    assert found
    return found


@pytest.mark.parametrize("pattern,groups", [(r"render_backward_kernelILi[124]E", 3), (r"render_backward_kernelILi8E", 2),
                                            (r"13render_kernelI", 3), (r"render_backward_rgb_kernel", 3)])
def test_workgroups_per_cu(kernels, pattern, groups):
    """256-thread workgroups: one wave of each on every SIMD."""
    hit = {k: v for k, v in kernels.items() if re.search(pattern, k)}
    assert hit
    for k, (lds, vgprs) in hit.items():
        assert groups * -(-lds // LDS_GRANULE) * LDS_GRANULE <= LDS_CU, (k, lds)
        assert groups * -(-vgprs // VGPR_GRANULE) * VGPR_GRANULE <= VGPRS_LANE, (k, vgprs)
