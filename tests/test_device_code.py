"""What the compiled kernels of libkvhot.so hold, read from their assembly."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import sea_module

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """The gfx950 instructions of every kernel of libkvhot.so, in order."""
    sea_module("_lib").load()
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    shutil.copy(sea_module("build").LIB_PATH, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out = []
    for f in sorted(d.iterdir()):
        if f.name.endswith("gfx950"):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", f.name], cwd=d, check=True,
                                  capture_output=True, text=True).stdout
            out += [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]
    assert out
    return out


def test_lds_dma_waits_for_m0(instructions):
    """gfx9: an LDS DMA may not directly follow a scalar write of M0, which
    holds its LDS address."""
    dma = [i for i, x in enumerate(instructions) if re.match(r"buffer_load.*\blds\b", x)]
    assert dma
    for i in dma:
        assert not re.match(r"s_\w+ m0,", instructions[i - 1]), instructions[i - 1:i + 1]
