"""The panels' matrix-core kernels as compiled (the assembly of csrc/panel.hip with the Makefile's flags), for what the
source relies on and cannot state:

* k_panel_gemm_h: no product takes as its starting sum the result of a product of another opcode.  The compiler puts
  no wait between two products that hand on exactly the same registers; across opcodes the second
  one can take the sum before the first one's result is there.
* k_panel_gemm: the barrier before a token tile's use waits until at most kCodeLoads vector loads are outstanding;
  that is the tile only if at least that many loads follow it.  Every path from a tile's last load into LDS
  to the next wait issues them, or the wait is for all loads."""
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


def waits_after(ins, start):
    """(loads issued since, outstanding allowed) at the next vector-memory wait on every path from `start`"""
    labels = {t[:-1]: i for i, t in enumerate(ins) if t.endswith(":")}
    found, seen, todo = [], set(), [(start, 0)]
    while todo:
        i, n = todo.pop()
        while i < len(ins) and (i, n) not in seen:
            seen.add((i, n))
            t = ins[i]
            m = re.search(r"vmcnt\((\d+)\)", t)
            if m:
                found.append((n, int(m.group(1))))
                break
            if "load_lds" in t:  # (the next tile's loads before any wait for this one)
                found.append((n, 63))
                break
            n += t.startswith(("global_load", "scratch_load"))
            if t.startswith("s_branch"):
                i = labels[t.split()[1]]
                continue
            if t.startswith("s_cbranch"):
                todo.append((labels[t.split()[1]], n))
            if t.startswith("s_endpgm"):
                found.append((n, 63))
                break
            i += 1
    return found


@pytest.mark.timeout(600)
def test_tile_waits_have_their_loads(kernels):
    src = (ca.PKG_DIR / "csrc" / "panel.hip").read_text()
    allowed = int(re.search(r"kCodeLoads = (\d+);", src).group(1))
    found = of(kernels, "k_panel_gemmI")
    assert len(found) == 10
    for name, ins in found.items():
        tiles = [i for i, t in enumerate(ins) if "load_lds" in t and not any("load_lds" in x for x in between(ins, i))]
        assert len(tiles) >= 6, name  # the first tile, four groups per trip, the remainders
        waits = [w for i in tiles for w in waits_after(ins, i + 1)]
        assert any(limit == allowed for _, limit in waits), name
        for n, limit in waits:
            assert limit == 0 or (limit <= allowed and n >= limit), (name, n, limit)


def between(ins, i):
    """the instructions from i to the next wait, barrier, load or branch"""
    for t in ins[i + 1:]:
        if t.startswith(("s_waitcnt", "s_barrier", "s_cbranch", "s_branch", "s_endpgm", "global_load_dword", "global_load_u")):
            if "load_lds" in t:
                yield t
            return
        yield t
