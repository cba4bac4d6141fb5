"""
What the compiler made of the device code, read from the library as it is built here.

Behind a block that only some lanes run, values are sometimes copied into accumulation registers before the other lanes are switched on again
(``s_or_b64 exec``): those lanes lose the value.  Two variants of kernels were compiled so, lost the upper addresses of their rows and ended in illegal memory
accesses.  It comes and goes with the pressure on the registers, so every build is looked at.
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


def lost_copies(listing):
    """
    :param listing: lines of ``llvm-objdump -d``
    :return: (kernel, instruction) of every copy into an accumulation register between the end of a masked block and the switch back
    """
    found, name, base, code, joins = [], None, 0, [], set()

    def look():
        at = {address: k for k, (address, _, _) in enumerate(code)}
        for join in joins:
            copies = []
            for _, op, args in code[at.get(join, len(code)) :]:
                if op.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                    break
                if op in ("s_or_b64", "s_mov_b64") and args.startswith("exec,"):
                    found.extend((name, c) for c in copies)
                    break
                if op == "v_accvgpr_write_b32" and re.search(r", v\d+$", args):
                    copies.append("%s %s" % (op, args))

    for line in listing:
        head = re.match(r"^([0-9a-f]{16}) <(.*)>:", line)
        if head:
            look()
            base, name, code, joins = int(head.group(1), 16), head.group(2), [], set()
            continue
        m = _LINE.match(line)
        if m:
            op, args, address, _, offset = m.groups()
            code.append((int(address, 16), op, (args or "").strip()))
            if op == "s_cbranch_execz":
                joins.add(base + int(offset or "0", 16))
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
