"""The kernels whose operands stream from HBM into LDS by direct loads order
those loads themselves: a wave whose LDS reads are still on their way at the
workgroup barrier could get bytes that another wave's next load has already
overwritten.  Checked on the built library: every barrier of these kernels
directly follows a wait for the wave's own LDS reads."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from rapidocrvl_amd import build

LLVM = os.path.join(build.ROCM, "llvm", "bin")
KERNELS = ("k_gemm_lds", "k_attn_prefill")


def _run(*cmd):
    return subprocess.run(cmd, check=True, capture_output=True, text=True).stdout


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instruction lists of the direct-load kernels, by symbol."""
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(build.LIB, d)
    _run(os.path.join(LLVM, "llvm-objdump"), "--offloading", lib)
    out = {}
    for obj in glob.glob(os.path.join(d, "*gfx950")):
        names = {n for n in re.findall(r"(_Z\w+)$", _run(os.path.join(LLVM, "llvm-readelf"), "-sW", obj), re.M)
                 if any(k in n for k in KERNELS)}
        if not names:
            continue
        text = _run(os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn",
                    "--disassemble-symbols=" + ",".join(sorted(names)), obj)
        for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
            name, body = part.split(">:", 1)
            out[name] = [ln.split("//")[0].strip() for ln in body.splitlines() if ln.strip()]
    return {n: code for n, code in out.items() if any("load_lds" in i for i in code)}


def test_barriers_wait_for_lds_reads(kernels):
    assert {k for k in KERNELS if any(k in n for n in kernels)} == set(KERNELS)
    for name, code in kernels.items():
        at = [i for i, ins in enumerate(code) if ins.startswith("s_barrier")]
        assert len(at) >= 2, name
        for i in at:
            assert re.match(r"s_waitcnt\b.*lgkmcnt\(0\)", code[i - 1]), (name, code[i - 1])
