"""Waits that the hardware needs and the compiler does not know of, in the sources and in the built library, without a GPU."""
import glob
import os
import re
import subprocess

import pytest

import _kernel_resources

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuv_amd", "csrc")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT = 2                                 # issue slots between the one instruction and the other


def _sources():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.hpp"))):
        with open(path) as f:
            yield os.path.basename(path), re.sub(r"//[^\n]*", "", f.read())


def _arguments(text, at):
    """The arguments of the call whose bracket opens at text[at]."""
    depth, args, start = 0, [], at + 1
    for i in range(at, len(text)):
        if text[i] in "([{":
            depth += 1
        elif text[i] in ")]}":
            depth -= 1
        if depth == 1 and text[i] == "," or depth == 0:
            args.append(text[start:i].strip())
            start = i + 1
        if depth == 0:
            return args


def test_wide_stores_with_a_scalar_offset_have_their_wait():
    """A buffer store of more than 8 bytes with a scalar offset reads its registers late: only buffer_store4 makes one, with a wait."""
    bare, waiting = [], 0
    for name, text in _sources():
        for m in re.finditer(r"raw_buffer_store_b(?:96|128)\(", text):
            offset = _arguments(text, m.end() - 1)[3]
            waits = re.match(r'[^;]*;\s*asm volatile\("s_nop 1" :: "v"\(v\)\);', text[m.end():]) is not None
            waiting += waits
            if offset != "0" and not waits:
                bare.append((name, offset))
    assert bare == [] and waiting == 1


def test_dpp_statements_begin_with_their_wait():
    """An operand that DPP reads across lanes must not have been written in the two preceding issue slots: a statement that the
    compiler cannot look into waits first."""
    bare, waiting = [], 0
    for name, text in _sources():
        macros = {m for m, body in re.findall(r"#define (\w+)(?:\([^)]*\))?((?:[^\n]*\\\n)*[^\n]*)", text) if "dpp" in body.lower()}
        for m in re.finditer(r"\basm(?: volatile)?\(", text):
            code = _arguments(text, m.end() - 1)[0]
            if "_dpp" in code or any(re.search(r"\b%s\b" % macro, code) for macro in macros):
                if re.match(r'"s_nop 1\\n\\t"', code):
                    waiting += 1
                else:
                    bare.append((name, code[:80]))
    assert bare == [] and waiting > 0


def test_loads_to_lds_have_their_wait():
    """A load's scalar operands must not have been written by a vector instruction in the five preceding issue slots: a statement waits
    for four behind its own write of M0."""
    bare, waiting = [], 0
    for name, text in _sources():
        for m in re.finditer(r"\basm(?: volatile)?\(", text):
            code = _arguments(text, m.end() - 1)[0]
            for macro, body in re.findall(r"#define (\w+) (.*)", text):
                code = re.sub(r"\b%s\b" % macro, lambda _: body, code)
            if re.search(r"(buffer|global)_load", code):
                if re.match(r's_mov_b32 m0, %0\\n\\ts_nop 3\\n\\t', code.replace('"', "")):
                    waiting += 1
                else:
                    bare.append((name, code[:80]))
    assert bare == [] and waiting > 0


_VECTOR = re.compile(r"v\[(\d+):(\d+)\]$|v(\d+)$")


def _registers(operand):
    m = _VECTOR.match(operand.split()[0]) if operand else None
    if m is None:
        return set()
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def _instructions(path):
    """(operation, operands) of every kernel, in the order of their addresses."""
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], capture_output=True, text=True, check=True).stdout
    for line in text.splitlines():
        if line.startswith("\t"):
            operation, _, operands = line.partition("//")[0].strip().partition(" ")
            if operation:
                yield operation, [o.strip() for o in operands.split(",")]


_SCALAR = re.compile(r"s\[(\d+):(\d+)\]$|s(\d+)$")


def _scalars(operand):
    m = _SCALAR.match(operand.split()[0]) if operand else None
    if m is None:
        return set()
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def _slots(operation, operands):
    return int(operands[0]) + 1 if operation == "s_nop" else 1


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    at = tmp_path_factory.mktemp("code")
    with open(_kernel_resources.LIBRARY, "rb") as f:
        data = f.read()
    found = []
    for i, elf in enumerate(_kernel_resources._code_objects(data)):
        path = at / ("%d.elf" % i)
        path.write_bytes(elf)
        found.append(list(_instructions(str(path))))
    assert found
    return found


def test_no_register_of_a_wide_store_is_written_early(library):
    stores = 0
    for code in library:
        for i, (operation, operands) in enumerate(code):
            if re.match(r"buffer_store_dwordx[34]", operation) is None or not operands[3].startswith("s"):
                continue
            stores += 1
            data, passed = _registers(operands[0]), 0
            for after, written in code[i + 1:i + 1 + WAIT]:
                if passed >= WAIT:
                    break
                assert not (after.startswith("v_") and _registers(written[0]) & data), (operation, operands, after, written)
                passed += _slots(after, written)
    assert stores > 0


def test_no_operand_of_dpp_is_written_late(library):
    broadcasts = 0
    for code in library:
        for i, (operation, operands) in enumerate(code):
            if not operation.endswith("_dpp"):
                continue
            broadcasts += 1
            source, passed = _registers(operands[1]), 0
            for before, written in reversed(code[max(0, i - WAIT):i]):
                if passed >= WAIT:
                    break
                passed += _slots(before, written) if before == "s_nop" else 0
                assert passed >= WAIT or not (before.startswith("v_") and _registers(written[0]) & source), (operation, operands, before, written)
                passed += before != "s_nop"
    assert broadcasts > 0


def test_no_operand_of_a_matrix_product_is_written_late(library):
    """Two slots here as well, where a statement of assembly makes the operand."""
    products = 0
    for code in library:
        for i, (operation, operands) in enumerate(code):
            if not operation.startswith("v_mfma"):
                continue
            products += 1
            source, passed = _registers(operands[1]) | _registers(operands[2]), 0
            for before, written in reversed(code[max(0, i - WAIT):i]):
                passed += _slots(before, written) if before == "s_nop" else 0
                if passed >= WAIT:
                    break
                assert not (before.startswith("v_") and not before.startswith("v_mfma") and _registers(written[0]) & source), (operation, operands, before, written)
                passed += before != "s_nop"
    assert products > 0


def test_no_scalar_operand_of_a_load_or_store_is_written_late(library):
    accesses, need = 0, 5
    for code in library:
        for i, (operation, operands) in enumerate(code):
            if re.match(r"(buffer|global)_(load|store|atomic)", operation) is None:
                continue
            source, passed = set().union(*(_scalars(o) for o in operands)), 0
            accesses += bool(source)
            for before, written in reversed(code[max(0, i - need):i]):
                passed += _slots(before, written) if before == "s_nop" else 0
                if passed >= need or not source:
                    break
                assert not (before.startswith("v_") and _scalars(written[0]) & source), (operation, operands, before, written)
                passed += before != "s_nop"
    assert accesses > 0
