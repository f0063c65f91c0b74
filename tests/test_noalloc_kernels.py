"""The kernels that gh_pcg_noalloc launches use no scratch memory: the runtime backs scratch
with device memory at the launch, and that solve promises to allocate none.  Read from the
metadata of the kernels in the built library (no GPU needed)."""
import re
import shutil
import struct
import subprocess

import pytest

from gridap_hip import _lib

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
# small_pcg_kernel by rows a thread, the CSR row kernels by lanes a row
EXPECTED = {"small_pcg_kernel": 4, "spmv_kernel": 4, "spmv_dir_kernel": 4, "update_zp_kernel": 1,
            "init_kernel": 1, "diag_inv_kernel": 1, "clear_stop_kernel": 1}


def device_objects(path):
    data = open(path, "rb").read()
    for m in re.finditer(re.escape(MAGIC), data):
        at = m.end()
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in name:
                yield data[m.start() + offset:m.start() + offset + size]


def test_no_scratch(tmp_path):
    if not shutil.which(READELF):
        pytest.skip("no llvm-readelf")
    scratch = {}
    for k, obj in enumerate(device_objects(_lib.LIB_PATH)):
        f = tmp_path / ("%d.o" % k)
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True,
                               check=True).stdout
        for kernel in re.split(r"\n  - (?=\.)", notes)[1:]:
            name = re.search(r"^\s*\.name:\s*(\S+)", kernel, re.M).group(1)
            size = re.search(r"\.private_segment_fixed_size:\s*(\d+)", kernel).group(1)
            stack = re.search(r"\.uses_dynamic_stack:\s*(\w+)", kernel)
            scratch[name] = int(size) if not stack or stack.group(1) == "false" else -1
    for kernel, count in EXPECTED.items():
        # the mangled name: <length><kernel> then the template arguments or the parameters
        found = {n: s for n, s in scratch.items() if "%d%sI" % (len(kernel), kernel) in n or
                 "%d%sE" % (len(kernel), kernel) in n}
        assert len(found) == count, (kernel, sorted(found))
        assert not any(found.values()), found
