"""
What the compiler made of the device code, read from the library as it is built here.

Where a block that only some lanes run has ended, values are sometimes copied into accumulation registers or scratch memory, or fetched back from there, before
the other lanes are switched on again: those lanes lose the value.  Three variants of kernels were compiled so; two lost the upper
addresses of their rows and ended in illegal memory accesses.  It comes and goes with the pressure on the registers, so every build is looked at.

What is looked at: the straight line of code from the end of a masked block -- where a branch past it leads, or behind the branch back of a loop that lanes leave one by
one -- to the switch back, be it that of an ``if``, of the change from ``if`` to ``else`` or of a loop.  What is not: ends with a branch in front of the switch, and moves between
ordinary registers, which are as often the block's own work.
"""

from __future__ import annotations

import os
import re
import struct
import subprocess

import pytest

from returnn_amd import build

OBJDUMP = os.path.join(os.path.dirname(build.ROCM_LIB_DIR), "lib", "llvm", "bin", "llvm-objdump")
_LINE = re.compile(r"^\t(\S+)(?: (.*?))?\s*// ([0-9A-F]{12}):(?:[^<]*<([^>+]+)(?:\+0x([0-9a-f]+))?>)?")


_COPY = re.compile(r"v_accvgpr_write_b32 a\d+, v\d+$|v_accvgpr_(read|mov)_b32 |scratch_(store|load)_")
_SWITCH_BACK = re.compile(r"s_(or|mov|xor)_b64 exec,|s_(or|andn2)_saveexec_b64 ")
_OTHER_SWITCH = re.compile(r"s_\w+_b64 exec,|s_\w+_saveexec_b64 |s_(cbranch|branch|endpgm|setpc)")


def lost_copies(listing):
    """
    :param listing: lines of ``llvm-objdump -d``
    :return: (kernel, instruction) of every copy between the end of a masked block and the switch back
    """
    found, name, base, code, ends = [], None, 0, [], set()

    def look():
        at = {address: k for k, (address, _) in enumerate(code)}
        starts = [at[end] for end in ends if end in at] + [k + 1 for k, (_, text) in enumerate(code) if text.startswith("s_cbranch_execnz")]
        for start in sorted(set(starts)):
            copies = []
            for _, text in code[start:]:
                if _SWITCH_BACK.match(text):
                    found.extend((name, c) for c in copies)
                    break
                if _OTHER_SWITCH.match(text):
                    break
                if _COPY.match(text):
                    copies.append(text)

    for line in listing:
        head = re.match(r"^([0-9a-f]{16}) <(.*)>:", line)
        if head:
            look()
            base, name, code, ends = int(head.group(1), 16), head.group(2), [], set()
            continue
        m = _LINE.match(line)
        if m:
            op, args, address, _, offset = m.groups()
            code.append((int(address, 16), "%s %s" % (op, (args or "").strip())))
            if op == "s_cbranch_execz":
                ends.add(base + int(offset or "0", 16))
    look()
    return found


def _code_objects(data):
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24 : entry + 24 + length]:
                yield data[at + offset : at + offset + size]
            entry += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


EXAMPLE = """
0000000000001000 <kernel>:
\ts_and_saveexec_b64 s[2:3], s[4:5]                          // 000000001000: BE822004
\ts_cbranch_execz 2                                          // 000000001004: BF880002 <kernel+0x10>
\tglobal_load_dword v3, v[6:7], off offset:64                // 000000001008: DC508040 037F0006
\tv_accvgpr_write_b32 a245, v15                              // 000000001010: D3D940F5 1800010F
\ts_or_b64 exec, exec, s[2:3]                                // 000000001018: 87FE027E
\tv_accvgpr_write_b32 a244, v14                              // 00000000101C: D3D940F4 1800010E
\ts_endpgm                                                   // 000000001024: BF810000
"""


def test_an_example_is_found():
    assert lost_copies(EXAMPLE.splitlines()) == [("kernel", "v_accvgpr_write_b32 a245, v15")]
    swapped = EXAMPLE.replace("a245, v15", "a245, s15")
    assert lost_copies(swapped.splitlines()) == []


# (what replaces the copy, the switch back and the branch of the example; whether it is a find)
FORMS = [
    ("v_accvgpr_write_b32 a245, v15", "s_or_b64 exec, exec, s[2:3]", None, True),
    ("v_accvgpr_read_b32 v15, a245", "s_mov_b64 exec, s[2:3]", None, True),
    ("scratch_store_dword off, v15, off offset:8", "s_or_saveexec_b64 s[2:3], s[2:3]", None, True),
    ("scratch_load_dword v15, off, off offset:8", "s_andn2_saveexec_b64 s[2:3], s[2:3]", None, True),
    ("v_accvgpr_write_b32 a245, v15", "s_xor_b64 exec, exec, s[2:3]", None, True),
    ("v_accvgpr_write_b32 a245, v15", "s_or_b64 exec, exec, s[2:3]", "loop", True),
    ("v_accvgpr_write_b32 a245, s15", "s_or_b64 exec, exec, s[2:3]", None, False),  # (the same for all lanes, and written again if need be)
    ("v_add_u32_e32 v15, 1, v15", "s_or_b64 exec, exec, s[2:3]", None, False),
    ("v_accvgpr_write_b32 a245, v15", "s_and_saveexec_b64 s[6:7], s[8:9]", None, False),  # (still inside: fewer lanes)
    ("v_accvgpr_write_b32 a245, v15", "s_branch 4", None, False),
]


@pytest.mark.parametrize("copy,switch,loop,find", FORMS)
def test_examples(copy, switch, loop, find):
    listing = EXAMPLE.replace("v_accvgpr_write_b32 a245, v15", copy).replace("s_or_b64 exec, exec, s[2:3]", switch)
    if loop:  # the load is the end of a loop that branches back
        listing = listing.replace("s_cbranch_execz 2  ", "s_nop 0  ").replace(" <kernel+0x10>", "")
        listing = listing.replace("global_load_dword v3, v[6:7], off offset:64                // 000000001008: DC508040 037F0006", "s_cbranch_execnz 65534 // 000000001008: BF89FFFE <kernel+0x4>")
    assert lost_copies(listing.splitlines()) == ([("kernel", copy)] if find else [])


def test_no_kernel_loses_a_copy(tmp_path):
    if not os.path.exists(build.LIB_PATH) or not os.path.exists(OBJDUMP):
        pytest.skip("no library or no llvm-objdump")
    with open(build.LIB_PATH, "rb") as f:
        objects = list(_code_objects(f.read()))
    assert len(objects) == build.TABLE_PARTS + 1
    running = []
    for k, code in enumerate(objects):
        path = tmp_path / ("%i.elf" % k)
        path.write_bytes(code)
        running.append(subprocess.Popen([OBJDUMP, "-d", str(path)], stdout=open(tmp_path / ("%i.s" % k), "w")))
    found, kernels = [], 0
    for k, process in enumerate(running):
        assert process.wait() == 0
        with open(tmp_path / ("%i.s" % k)) as f:
            lines = f.readlines()
        kernels += sum("k_lstm2_" in line for line in lines if line.endswith(">:\n"))
        found += lost_copies(lines)
    assert kernels > 100 and not found, found
