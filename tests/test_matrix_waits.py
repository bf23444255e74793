"""Every result of a matrix instruction in the built libraries is waited for before anything but the next product's sum touches it.  The hardware does
not hold such an instruction back; the compiler counts instructions and inserts the rest as `s_nop`, and has left that out where paths meet: in an earlier form of
the delta rule's scan (csrc/qmk_hybrid_chunks.h) a product's result was moved two instructions behind it, at one number of tiles a wave, unless `settle` held it.  So this walks all paths of every kernel
with a matrix instruction, as built."""
import re
import subprocess
from pathlib import Path

import pytest

from conftest import ROOT
from test_kernel_resources import device_code

LIBRARIES = ("libqmk_hip.so", "libqmk_hybrid.so")
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
#: instructions between a product and the first use of its result, but as the next product's sum (CDNA ISA guide, manually inserted wait states: eight passes of a
#: single-precision product, four of a bf16 one; the shortest distance that the compiler leaves within one block is the same)
WAIT = {"v_mfma_f32_16x16x4_f32": 10, "v_mfma_f32_16x16x16_bf16": 8, "v_mfma_f32_16x16x32_bf16": 8}
REGISTER = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")


def registers(text):
    found = set()
    for kind, one, low, high in REGISTER.findall(text):
        found.update((kind, i) for i in range(int(one or low), int(one or high) + 1))
    return frozenset(found)


def kernels(listing):
    """{name: [(address, label or None, operation, operands)]} of a disassembly with symbolized branches."""
    found, name, label = {}, None, None
    for line in listing.splitlines():
        if line.startswith("<"):
            mark = line[1 : line.index(">")]
            if re.fullmatch(r"L\d+", mark):
                label = mark
            else:
                name, label = mark, None
                found[name] = []
        elif line.startswith("\t") and name and "//" in line:
            code, _, note = line.strip().partition("//")
            operation, _, operands = code.strip().partition(" ")
            found[name].append((int(note.split(":")[0], 16), label, operation, operands.strip()))
            label = None
    return found


def unwaited(code):
    """(instruction, its operands, instructions still to wait) of every use that comes too early on some path."""
    labels = {label: i for i, (_, label, _, _) in enumerate(code) if label}
    place = {address: i for i, (address, *_) in enumerate(code)}
    starts, follow = {0, *labels.values()}, {}
    for i, (_, _, op, args) in enumerate(code):
        if op.startswith("s_cbranch"):
            follow[i] = [i + 1, labels[args.split()[0]]]
        elif op == "s_branch":
            follow[i] = [labels[args.split()[0]]]
        elif op == "s_setpc_b64":           # a far jump: s_getpc, an offset from the next instruction on, its upper half
            assert code[i - 3][2] == "s_getpc_b64" and code[i - 2][2] == "s_add_u32"
            follow[i] = [place[code[i - 2][0] + int(code[i - 2][3].split(",")[2], 0)]]
        elif op == "s_endpgm":
            follow[i] = []
        else:
            assert op not in ("s_swappc_b64", "s_call_b64", "s_cbranch_g_fork"), op
            continue
        starts.update(follow[i] + [i + 1])
    parsed = {}
    for i, (_, _, op, args) in enumerate(code):
        if op.startswith("v_mfma"):
            to, a, b = (registers(part) for part in args.split(",")[:3])
            parsed[i] = (WAIT[op], to, a | b)
        elif op == "s_nop":
            parsed[i] = (int(args, 0) + 1, None, frozenset())
        else:
            parsed[i] = (1, None, registers(args))
    early, state, work = set(), {0: {}}, [0]
    while work:
        i = work.pop()
        waits = dict(state[i])
        while True:
            count, result, used = parsed[i]
            if waits:
                early.update((code[i][2], code[i][3], waits[r]) for r in used if r in waits)
                passed = 1 if result else count
                waits = {r: left - passed for r, left in waits.items() if left > passed}
            if result:
                waits.update(dict.fromkeys(result, count))
            ends = i in follow
            targets = follow[i] if ends else [i + 1]
            if ends or i + 1 in starts:
                break
            i += 1
        for t in targets:
            if t >= len(code):
                continue
            known = state.get(t)
            if known is None:
                state[t] = dict(waits)
                work.append(t)
            else:
                longer = {r: left for r, left in waits.items() if left > known.get(r, 0)}
                if longer:
                    known.update(longer)
                    work.append(t)
    return early


@pytest.mark.parametrize("library", LIBRARIES)
def test_results_are_waited_for_on_every_path(tmp_path, library):
    path = ROOT / "qimeng-megakernel_amd" / library
    if not path.is_file() or not OBJDUMP.is_file():
        pytest.skip("needs the built library and llvm-objdump")
    checked = 0
    for i, object_code in enumerate(device_code(path.read_bytes())):
        (tmp_path / f"{i}.co").write_bytes(object_code)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", tmp_path / f"{i}.co"], capture_output=True, text=True, check=True).stdout
        for name, code in kernels(listing).items():
            if any(op.startswith("v_mfma") for _, _, op, _ in code):
                early = unwaited(code)
                assert not early, (name, sorted(early)[:4])
                checked += 1
    assert checked > 5


PRODUCT = "v_mfma_f32_16x16x4_f32 a[0:3], v1, v2, a[0:3]"


@pytest.mark.parametrize("lines,found", [
    ([PRODUCT, "s_nop 9", "v_accvgpr_read_b32 v3, a0"], False),
    ([PRODUCT, "s_nop 8", "v_accvgpr_read_b32 v3, a3"], True),
    ([PRODUCT, PRODUCT, "s_nop 9", "ds_write_b128 v9, a[0:3]"], False),
    (["s_cbranch_scc1 L0", PRODUCT, "<L0>:", "s_nop 7", "v_mov_b32_e32 a1, v0"], True),             # on the path that does not jump
    (["<L0>:", "v_accvgpr_mov_b32 a8, a2", "s_nop 3", PRODUCT, "s_cbranch_scc1 L0"], True),         # round a loop
    (["<L0>:", "s_nop 9", "v_accvgpr_mov_b32 a8, a2", "s_nop 3", PRODUCT, "s_cbranch_scc1 L0"], False),
    ([PRODUCT, "s_nop 4", "v_mfma_f32_16x16x4_f32 a[4:7], v1, a2, a[4:7]"], True),
], ids=["waited", "one short", "sum", "branch", "loop", "loop, waited", "operand"])
def test_the_walk_finds_what_is_too_early(lines, found):
    text, address = ["<kernel>:"], 0x100
    for line in lines + ["s_endpgm"]:
        text.append(line if line.startswith("<") else f"\t{line}    // {address:012X}: 00000000")
        address += 4
    assert bool(unwaited(kernels("\n".join(text))["kernel"])) == found
