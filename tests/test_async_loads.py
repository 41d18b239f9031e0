"""The compiler believes a register that an inline assembly load fills to be valid at once: the assembly of the kernels with such
loads is followed from every load along every path, and nothing may touch its registers before a wait that covers it."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tuna_amd", "csrc")
REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _registers(text):
    return frozenset((f, r) for f, lo, hi, one in REG.findall(text) for r in range(int(lo or one), int(hi or one) + 1))


def _functions(text):
    """(name, [(instruction or 'label:', inside inline assembly)]) of every kernel."""
    name, body, inside = None, [], False
    for line in text.splitlines():
        if m := re.match(r"(_Z\w+):", line):
            name, body, inside = m.group(1), [], False
        elif line.startswith(".Lfunc_end") and name:
            yield name, body
            name = None
        elif "ASMSTART" in line or "ASMEND" in line:
            inside = "ASMSTART" in line
        elif m := re.match(r"(\.LBB\w+:)", line):
            body.append((m.group(1), False))
        elif name and (line := line.split(";")[0].strip()) and not line.startswith("."):
            body.append((line, inside))


def _follow(body):
    """(number of inline assembly loads into registers, [(load, instruction that touches its registers too early)])"""
    label = {t[:-1]: i for i, (t, _) in enumerate(body) if t.endswith(":")}
    seen, todo, early, loads = set(), [(0, ())], set(), set()
    while todo:
        # pending: the wave's vector memory operations from the oldest such load on; they end in order
        i, pending = todo.pop()
        while i < len(body):
            text, inside = body[i]
            op = text.split()[0]
            if text.endswith(":"):
                if (i, pending) in seen:
                    break
                seen.add((i, pending))
            elif op == "s_waitcnt":
                if m := re.search(r"vmcnt\((\d+)\)", text):
                    pending = pending[max(0, len(pending) - int(m.group(1))):]
                    while pending and not pending[0][1]:
                        pending = pending[1:]
            elif op == "s_endpgm":
                break
            elif op == "s_branch":
                i = label[text.split()[1]]
                continue
            else:
                assert op not in ("s_setpc_b64", "s_swappc_b64"), text
                if pending:
                    regs = _registers(text)
                    early.update((body[p][0], text) for p, held in pending if held & regs)
                if op.startswith("s_cbranch"):
                    todo.append((label[text.split()[1]], pending))
                if re.match("(buffer|global|flat|scratch)_(load|store|atomic)", op):
                    held = frozenset()
                    if inside and "_load" in op and not text.endswith(" lds"):
                        held = _registers(text.split(",")[0])
                        loads.add(i)
                    if held or pending:
                        pending += ((i, held),)
            i += 1
    return len(loads), sorted(early)


@pytest.mark.parametrize("source,kernels", [("gemm_wide.hip", 3)])
def test_nothing_touches_a_register_on_its_way(tmp_path, source, kernels):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    with open(os.path.join(CSRC, "Makefile")) as f:
        flags = re.search(r"^HIPFLAGS \?= ((?:.*\\\n)*.*)", f.read(), re.M).group(1).replace("\\\n", " ").replace("$(ARCH)", "gfx950")
    out = tmp_path / "kernels.s"
    subprocess.run([hipcc, *flags.split(), "--offload-device-only", "-S", source, "-o", str(out)], cwd=CSRC, check=True, capture_output=True)
    found = 0
    for name, body in _functions(out.read_text()):
        loads, early = _follow(body)
        assert not early, (name, early[:4])
        found += loads > 0
    assert found == kernels
