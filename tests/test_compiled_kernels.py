"""The compiled kernels of the built library: memory ordering that no run can
show reliably, read from the gfx950 code."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from wabbit_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = os.path.join(build.PKG, build.LIBNAME)
    if not os.path.exists(lib):
        build.build(False)
    at = str(tmp_path_factory.mktemp("code"))
    subprocess.run([OBJDUMP, "--offloading", shutil.copy(lib, at)], check=True, capture_output=True)
    return [f for f in glob.glob(os.path.join(at, "*gfx950")) if os.path.getsize(f)]


def _kernels(code_objects, name):
    """{symbol: instructions} of the kernels whose mangled names hold `name`"""
    out = {}
    for obj in code_objects:
        table = subprocess.run([OBJDUMP, "-t", obj], check=True, capture_output=True, text=True).stdout
        for sym in re.findall(rf"F \.text\s+\S+(?: \.protected)? (\S*{name}\S*)", table):
            text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={sym}", obj], check=True, capture_output=True,
                                  text=True).stdout
            out[sym] = [m.group(1) for m in re.finditer(r"^\s+([a-z]\w+ ?[^/\n]*)", text, re.M)]
    return out


def test_last_workgroup_of_the_dt_acquires_what_the_others_released(code_objects):
    """The workgroup that counts itself the last of a dt launch reads the
    minimum that the others added.  They release it through the counter, so an
    acquire (buffer_inv) has to follow the counting add before the minimum is
    taken (the swap)."""
    kernels = _kernels(code_objects, "4k_dtILi")
    assert len(kernels) == 4
    for sym, ins in kernels.items():
        count = [i for i, x in enumerate(ins) if x.startswith("global_atomic_add_x2")]
        take = [i for i, x in enumerate(ins) if x.startswith("global_atomic_swap_x2")]
        assert len(count) == 1 and len(take) == 1 and count[0] < take[0], sym
        release = [x for x in ins[:count[0]] if x.startswith("buffer_wbl2")]
        between = ins[count[0] + 1:take[0]]
        assert release and any(x.startswith("buffer_inv") for x in between), (sym, between)
