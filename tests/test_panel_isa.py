"""The panels' matrix-core kernels as compiled (the assembly of csrc/panel.hip with the Makefile's flags), for what the
source relies on and cannot state:

* k_panel_gemm_h: no product takes as its starting sum the result of a product of another opcode.  The compiler puts
  no wait between two products that hand on exactly the same registers; across opcodes the second
  one can take the sum before the first one's result is there."""
import re
import shlex
import subprocess
from collections import defaultdict

import pytest

import chpe_amd as ca


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """kernel name -> its instructions (labels kept), from the compile command that make would run"""
    out = subprocess.run(["make", "-n", "-B", "_build/panel.o"], cwd=ca.PKG_DIR, capture_output=True, text=True, check=True).stdout
    cmd = shlex.split(next(ln for ln in out.splitlines() if "panel.hip" in ln and "-c" in ln))
    asm = tmp_path_factory.mktemp("isa") / "panel.s"
    cmd[cmd.index("-o") + 1] = str(asm)
    cmd[cmd.index("-c")] = "-S"
    subprocess.run(cmd + ["--cuda-device-only", "-w"], cwd=ca.PKG_DIR, check=True)
    ins, name = defaultdict(list), None
    for line in asm.read_text().splitlines():
        m = re.match(r"(_ZN\S+):", line)
        if m:
            name = m.group(1)
        elif line.startswith("\t.section"):
            name = None
        elif name:
            t = line.split(";")[0].strip()
            if t and (not t.startswith(".") or t.endswith(":")):
                ins[name].append(t)
    return ins


def of(kernels, pattern):
    found = {n: v for n, v in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    return found


MFMA = re.compile(r"(v_mfma_\w+) ([va]\[\d+:\d+\]), .*, (\S+)$")


@pytest.mark.timeout(600)
def test_products_start_from_their_own_opcode(kernels):
    for name, ins in of(kernels, "k_panel_(gemm|attn)").items():
        n = 0
        last = {}  # result registers -> the opcode of the product that wrote them last
        for t in ins:
            m = MFMA.match(t)
            if m:
                op, dst, start = m.groups()
                n += 1
                assert last.get(start, op) == op, (name, t)
                last[dst] = op
            elif t.startswith("v_") and " v[" in t:
                last.pop(t.split()[1].rstrip(","), None)
        assert n > 0, name
