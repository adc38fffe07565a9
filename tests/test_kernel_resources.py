"""Registers and LDS of the built kernels against what their launch rules
assume: the workgroups per CU that a kernel's template arguments name have to
fit, or the grid runs in two rounds (CPU; reads the built code objects)."""
import re
import shutil
import struct
import subprocess

import pytest

from gcge_old_amd import _native

ROCM_BIN = "/opt/rocm/llvm/bin:/opt/rocm/lib/llvm/bin"
SIMD_VGPRS, CU_LDS = 512, 160 * 1024  # registers per lane of a SIMD, LDS bytes of a CU


def _code_objects(data):
    """The gfx950 code objects in the offload bundles of a library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        pos = at + len(magic)
        count, = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if size and b"gfx950" in target:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + len(magic))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: {resource: value}} from the metadata of the code objects."""
    readelf, demangle = shutil.which("llvm-readelf", path=ROCM_BIN), shutil.which("c++filt")
    with open(_native.lib_path("libgcge_hip.so"), "rb") as f:
        data = f.read()
    found = {}
    for i, blob in enumerate(_code_objects(data)):
        path = tmp_path_factory.mktemp("code") / f"{i}.elf"
        path.write_bytes(blob)
        notes = subprocess.run([readelf, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for entry in re.split(r"^  - (?=\.agpr_count|\.args)", notes, flags=re.M)[1:]:
            symbol = re.search(r"\.symbol:\s+'?(\S+?)\.kd", entry).group(1)
            found[symbol] = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)$", entry, flags=re.M)}
    names = subprocess.run([demangle], input="\n".join(found), capture_output=True, text=True, check=True).stdout
    return dict(zip(names.split("\n"), found.values()))


def test_gram_workgroups_fit(kernels):
    """The last template argument of k_gram_wide is the number of workgroups
    per CU that its grid is made for."""
    instances = {n: r for n, r in kernels.items() if re.search(r"\bk_gram_wide<", n)}
    assert len(instances) >= 40
    for name, r in instances.items():
        blocks = int(re.search(r"k_gram_wide<[^>]*\b(\d+)>", name).group(1))
        waves_per_simd = SIMD_VGPRS // (-(-r["vgpr_count"] // 8) * 8)
        waves = r["max_flat_workgroup_size"] // 64
        assert r["vgpr_spill_count"] == 0, name
        assert blocks in (1, 2) and waves_per_simd * 4 >= blocks * waves, (name, r)
        assert blocks * r["group_segment_fixed_size"] <= CU_LDS, (name, r)
