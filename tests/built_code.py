"""The gfx950 code of the built library, kernel by kernel (for the tests of what
the compiler made of the sources): hipcc's offload bundles taken apart and
disassembled with the ROCm LLVM tools."""
import glob
import os
import re
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

from capi_types import LIB, REPO

sys.path.insert(0, os.path.join(REPO, "flash-attention-sm75-register-fused_amd"))
import build_native  # noqa: E402

LLVM = os.path.join(build_native.ROCM, "llvm", "bin")


def _code_object(path):
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", path],
                           capture_output=True, text=True, check=True).stdout
    asm = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", path],
                         capture_output=True, text=True, check=True).stdout
    vgprs = {}
    for kernel in re.split(r"\n  - (?=\.)", notes)[1:]:
        name = re.search(r"\n    \.name:\s+(\S+)", kernel)
        # (accumulation registers share the allocation, after the others)
        count, acc = (re.search(rf"\.{c}_count:\s+(\d+)", kernel) for c in ("vgpr", "agpr"))
        if name and count:
            vgprs[name.group(1)] = int(count.group(1)) - (int(acc.group(1)) if acc else 0)
    found = []
    for part in re.split(r"\n(?=[0-9a-f]+ <_ZN2fa\S+>:)", asm)[1:]:
        name = re.match(r"[0-9a-f]+ <(\S+)>:", part).group(1)
        lines = [line.split("//")[0].strip() for line in part.split("\n")[1:]]
        if name in vgprs:
            found.append((name, vgprs[name], [line for line in lines if line]))
    assert len(found) == len(vgprs), (path, sorted(set(vgprs) - {f[0] for f in found}))
    return found


def kernels():
    """(mangled name, vector registers without accumulation ones, instructions) of every
    kernel of the library."""
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built: run __graft_entry__.build()")
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("the ROCm LLVM tools are not available")
    tmp = tempfile.mkdtemp(prefix="fa_built_code_")
    try:
        lib = shutil.copy(LIB, tmp)
        subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], cwd=tmp,
                       capture_output=True, check=True)
        objects = sorted(glob.glob(lib + ".*gfx950"))
        with ThreadPoolExecutor(8) as pool:
            return [k for found in pool.map(_code_object, objects) for k in found]
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
