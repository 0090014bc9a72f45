"""Products written as assembly (mfma32_new, mfma32_onto and the like) are not known to the compiler as products: it inserts no wait states between one
and who uses its result.  The generated code of the kernels that have them keeps the distances by the order of their work; here they are counted (CPU:
compiles to assembly, runs nothing)."""
import re
import subprocess

import pytest

BEHIND = 19    # wait states from a 32x32 product of 16-bit operands to another use of its result
IN_FRONT = 2   # from a vector instruction's result to a product that reads it
PRODUCT = 8    # wait states that a product in between takes at least


def _registers(operand):
    m = re.fullmatch(r"-?([va])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    if not m:
        return set()
    first, last = (m[2], m[3]) if m[2] else (m[4], m[4])
    return {(m[1], r) for r in range(int(first), int(last) + 1)}


def _kernels(text):
    """(name, [(opcode, operands, by hand)], {label: index}) of every kernel."""
    for m in re.finditer(r"\n(_ZN\S*kernel\S*):[^\n]*\n(.*?)\n\s*s_endpgm", text, re.S):
        code, labels, by_hand = [], {}, False
        for line in map(str.strip, m[2].splitlines()):
            if "#ASMSTART" in line or "#ASMEND" in line:
                by_hand = "#ASMSTART" in line
            elif label := re.match(r"(\.LBB\d+_\d+):", line):
                labels[label[1]] = len(code)
            elif line and line[0] not in ";.":
                op, _, rest = line.split(";")[0].strip().partition(" ")
                code.append((op, [o.strip() for o in rest.split(",")], by_hand))
        yield m[1], code, labels


def _behind(code, labels, start, limit):
    """Instructions reached within `limit` wait states behind `start` on any path, with the least distance."""
    def next_of(n):
        op, operands, _ = code[n]
        jump = [labels[operands[0]]] if op.startswith(("s_cbranch", "s_branch")) and operands[0] in labels else []
        return [k for k in jump + ([] if op == "s_branch" else [n + 1]) if k < len(code)]
    nearest, todo = {}, [(k, 0) for k in next_of(start)]
    while todo:
        n, waited = todo.pop()
        if waited >= limit or nearest.get(n, limit) <= waited:
            continue
        nearest[n] = waited
        op, operands, _ = code[n]
        waited += PRODUCT if op.startswith("v_mfma") else int(operands[0]) + 1 if op == "s_nop" else 1
        todo += [(k, waited) for k in next_of(n)]
    return nearest


@pytest.mark.parametrize("source", ["attn_fwd_pipe", "attn_bwd_pipe"])
def test_wait_states_around_products_by_hand(source, tmp_path):
    from odysseus_transformer_amd import build
    out = tmp_path / "kernels.s"
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "-I", str(build.INCLUDE), "-S", "--cuda-device-only", str(build.CSRC / f"{source}.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    products = 0
    for name, code, labels in _kernels(out.read_text()):
        for n, (op, operands, by_hand) in enumerate(code):
            if op.startswith("v_mfma") and by_hand:
                products += 1
                result = _registers(operands[0])
                for k, waited in _behind(code, labels, n, BEHIND).items():
                    other, those, _ = code[k]
                    if other.startswith("v_mfma") and _registers(those[0]) == result and not (_registers(those[1]) | _registers(those[2])) & result:
                        continue   # the next product of the same sum
                    assert not set().union(*map(_registers, those)) & result, f"{name}: {other} {those} {waited} wait states behind {op} {operands}"
            elif op.startswith("v_") and not op.startswith("v_mfma"):
                result = _registers(operands[0])
                for k, waited in _behind(code, labels, n, IN_FRONT).items() if result else ():
                    other, those, hand = code[k]
                    assert not (hand and other.startswith("v_mfma") and set().union(*map(_registers, those[1:])) & result), f"{name}: {other} {those} {waited} behind {op} {operands}"
    assert products > 50
