"""Wait states behind matrix instructions in the built kernels, read from the assembly of the library's own gfx950 code objects.

A vector or memory instruction must not touch the result of a matrix instruction before some wait states have passed; the hardware does not
look.  The compiler inserts them, but where paths join again behind a condition it follows only one of them back to the product: one that
jumps over the code between the two may come too early (seen: a score of the step before, 1 state of 8).  Here every path is followed."""
import os
import re
import subprocess

import pytest

from test_registers_cpu import _sections
from turbodeberta_amd import _build, _lib

REGISTERS = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")
# States that the compiler leaves in straight code before a result is read (before it is overwritten: one less, bar the last).
STATES = {"16x16x32": 8, "32x32x16": 12, "16x16x4": 10}
MOST = 12


def _registers(text):
    found = set()
    for first, last, one in REGISTERS.findall(text):
        found.update([int(one)] if one else range(int(first), int(last) + 1))
    return found


def _touched(line):
    """(registers read, registers written) of a vector, memory or LDS instruction."""
    op, _, rest = line.partition(" ")
    first, _, others = rest.partition(",")
    if op.startswith("v_cmp") or re.match(r"(ds_write|ds_add|(global|buffer|flat|scratch)_(store|atomic))", op):
        return _registers(rest), set()
    if op.startswith("v_permlane") and "swap" in op:
        return _registers(rest), _registers(rest)
    return _registers(others), _registers(first)


def early_uses(code):
    """code: [(address, text, target of a branch or None)].  Uses of a product's result that a path reaches too early, as
    (product, user, states passed, states needed)."""
    index = {address: i for i, (address, _, _) in enumerate(code)}
    branch = [i for i, (_, text, _) in enumerate(code) if text.startswith(("s_cbranch", "s_branch"))]
    near, at = set(), 0
    for i in range(len(code)):              # (a branch within MOST instructions: straight code is the compiler's own affair)
        while at < len(branch) and branch[at] < i:
            at += 1
        if at < len(branch) and branch[at] <= i + MOST:
            near.add(i)
    touched, bad = {}, []
    for start in sorted(near):
        text = code[start][1]
        if not text.startswith("v_mfma"):
            continue
        shape = next(s for s in STATES if s + "_" in text)
        need, seen = STATES[shape], {}
        paths = [(start + 1, 0, frozenset(_registers(text.split(",")[0])))]
        while paths:
            i, passed, live = paths.pop()
            while i < len(code) and passed < need and live and seen.get(i, MOST) > passed:
                seen[i] = passed
                text, target = code[i][1:]
                op = text.split(" ", 1)[0]
                if op.startswith("v_mfma"):
                    a, b, c = (_registers(part) for part in text.split(",")[1:4])
                    if live & (a | b):
                        bad.append((code[start][1], text, passed, need))
                        break
                    live -= c | _registers(text.split(",")[0])          # (in order behind it, whose own result then counts)
                elif not op.startswith("s_"):
                    if i not in touched:
                        touched[i] = _touched(text)
                    reads, writes = touched[i]
                    if live & reads or (live & writes and passed < need - (shape != "16x16x4")):
                        bad.append((code[start][1], text, passed, need))
                        break
                    live -= writes
                passed += int(text.split()[1]) + 1 if op == "s_nop" else 1
                if op.startswith("s_cbranch"):
                    paths.append((index[target], passed, live))
                elif op == "s_branch":
                    i = index[target]
                    continue
                elif op.startswith(("s_endpgm", "s_setpc")):
                    break
                i += 1
    return bad


def _kernels(tmp_path):
    tool = os.path.join(os.path.dirname(os.path.realpath(_build.hipcc())), "..", "llvm", "bin", "llvm-objdump")
    fat = dict(_sections(open(_lib.LIB_PATH, "rb").read()))[b".hip_fatbin"]
    for at in [m.start() for m in re.finditer(rb"\x7fELF", fat)]:
        if b".note" not in dict(_sections(fat[at:])):
            continue
        path = tmp_path / f"{at}.o"
        path.write_bytes(fat[at:])
        name, code = None, []
        for line in subprocess.run([tool, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout.splitlines():
            if m := re.match(r"[0-9a-f]+ <(\S+)>:", line):
                if code:
                    yield name, code
                name, code = m.group(1), []
            elif m := re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):(?:.*<\S+?(?:\+0x([0-9a-f]+))?>)?", line):
                target = m.group(1).startswith(("s_cbranch", "s_branch"))
                code.append((int(m.group(2), 16), m.group(1), int(m.group(3) or "0", 16) if target else None))
        if code:
            yield name, code


def test_results_are_there_on_every_path(tmp_path):
    _lib.load()
    kernels, early = 0, {}
    for name, code in _kernels(tmp_path):
        start = code[0][0]
        code = [(address - start, text, target) for address, text, target in code]
        kernels += any(text.startswith("v_mfma") for _, text, _ in code)
        if found := early_uses(code):
            early[name] = found
    assert kernels > 100
    assert not early, "\n".join(f"{name}: {u}" for name, uses in early.items() for u in uses)


@pytest.mark.parametrize("skipped,found", [(0, 1), (1, 0)])
def test_a_path_that_comes_too_early_is_found(skipped, found):
    """Behind a branch that jumps over ten instructions: the product's result one state after the jump, or after all that is needed."""
    code = [(0, "v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], 0", None), (8, "s_cbranch_scc1 5", 100)]
    code += [(12 + 8 * i, f"v_add_f32_e32 v{20 + i}, v40, v41", None) for i in range(10)]
    code += [(100, f"s_nop {7 * skipped}", None), (104, "v_add_f32_e32 v12, v2, v13", None), (108, "s_endpgm", None)]
    assert len(early_uses(code)) == found
