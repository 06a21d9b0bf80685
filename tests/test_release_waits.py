"""Releases in the code built for gfx950 (read from the libraries' own device code, on the CPU): the write-back of the
L2 is waited for before anything after it. The compiler leaves that wait out where it knows of no other memory
operation on its way, so every release has to bring its own."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LIBRARIES = ["gpu_workgroup_managment_amd/libwgm.so", "tests/kernel_merge/libwgm_kmerge.so",
             "tests/kernels/libwgm_userk.so"]
# HIP's own grid barrier, a reference point: its fences come from HIP's headers, and it guards no data
NOT_OURS = "k_coop_barrier"
MEMORY = re.compile(r"^(global|flat|buffer|scratch|s_barrier|s_branch|s_cbranch|s_endpgm|s_setpc)")


def device_code(library, tmp_path):
    (tmp_path / "lib.so").symlink_to(os.path.join(ROOT, library))
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    for f in sorted(tmp_path.glob("lib.so.*gfx950")):
        yield subprocess.run([OBJDUMP, "-d", f], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("library", LIBRARIES)
def test_release_waits_for_the_write_back(library, tmp_path):
    if not os.path.exists(os.path.join(ROOT, library)):
        pytest.skip(f"{library} is not built")
    releases, bare, kernel, waiting = 0, [], "", False
    for text in device_code(library, tmp_path):
        for line in text.split("\n"):
            head = re.match(r"^[0-9a-f]+ <(.*)>:", line)
            if head:
                kernel, waiting = head.group(1), False
                continue
            op = line.strip()
            if op.startswith("buffer_wbl2"):
                releases += 1
                waiting = NOT_OURS not in kernel
            elif waiting and op.startswith("s_waitcnt") and "vmcnt(0)" in op:
                waiting = False
            elif waiting and MEMORY.match(op):
                bare.append(f"{kernel}: {op.split('//')[0].strip()}")
                waiting = False
    assert releases > 0
    assert not bare, bare[:5]
